// Banded factorization without pivoting in FP64 (see fem_lu.hpp).
//
// The operator is symmetric (its lower triangle mirrored), so the elimination runs on the lower triangle only
// (LDL^T) and writes the LU form the solves read: L (unit lower) below the diagonal, U = D L^T on and above it.
// Row c of U is column c of the eliminated lower triangle, the value the elimination divides by the pivot.
// Right-looking, by panels of kLuPanel columns, one launch per panel. For panel [k0, k1), its diagonal block eliminated
// (for the first panel by a launch of its own, for the others by the first workgroup of the launch before), every 64 x 64
// lower output tile of the trailing block a(i, j), i >= j in [k1, k1 + bw),
//   1. eliminates the 64 or 128 panel rows it needs against that block: l(i, c) and u(c, i), into LDS;
//   2. takes a(i, j) -= L21 U12; the tiles on the diagonal write U12 to the upper band. The raw rows stay in the lower
//      band, where every tile reads them, and L = (U / pivots)^T takes their place in one pass after the last panel.
// At bandwidths in the hundreds a launch is a chain of latencies (loads, 32 eliminations of a row, the product, 32 of the
// next diagonal block), hardly work, so repeating the rows' elimination in every tile costs less than a launch of its own
// for it: 3,240 DOFs at bandwidth 356 take 11.0 us a panel, against 15.4 + 20.5 us with rows and update apart. Factor
// alone, rows and update apart against this: 6.8 and 2.3 ms at 6,069 x 923, 8.6 and 3.1 at 7,581 x 1,142, 14.5 and 7.1 at
// 13,125 x 1,952, 18.3 and 13.3 at 12,288 x 3,170, 33.3 and 29.0 at 11,616 x 5,942, 210 and 210 at 22,326 x 11,348.
// Each entry takes the column-by-column updates in the same order as the column form of the restated reference
// solver, with the panel's updates of the trailing block summed before they are applied: results agree with
// unblocked LU to rounding.
//
// Substitution: the 64 x 64 diagonal blocks of L and U are inverted once per factorization. A solve walks the
// rows in blocks of 64: the block's products with the entries solved before it (up to bw per row) as an LDS-tiled
// product over 64-entry tiles (the next tile prefetched into registers), then the block's triangle as a product
// with its inverse. One workgroup per 16 (or 4) right-hand sides, or per column at narrow bands; sums in a fixed order.
#include "fem_lu.hpp"
#include "fem_kernels.hpp"
#include "fem_reduce.hpp"

#include <algorithm>
#include <stdexcept>

namespace femgpu {

namespace {

constexpr int kLuPanel = 32;
constexpr int kTile = 64;
using v2u = uint32_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ double& at(double* ab, int64_t ld, int bw, int64_t i, int64_t j) {
    return ab[i * ld + (j - i + bw)];
}
__device__ __forceinline__ double atc(const double* ab, int64_t ld, int bw, int64_t i, int64_t j) {
    return ab[i * ld + (j - i + bw)];
}

__global__ __launch_bounds__(256) void band_zero_kernel(double* __restrict__ ab, int64_t count) {
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < count; t += (int64_t)gridDim.x * blockDim.x)
        ab[t] = 0.0;
}

// One thread per block: its 9 values into the band.
__global__ __launch_bounds__(256) void band_fill_kernel(double* __restrict__ ab, int64_t ld, int bw,
                                                        int64_t num_blocks, const int* __restrict__ blk_row,
                                                        const int* __restrict__ colidx,
                                                        const double* __restrict__ S) {
    const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (k >= num_blocks) return;
    const int64_t I = blk_row[k], J = colidx[k];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) at(ab, ld, bw, 3 * I + r, 3 * J + c) = S[9 * k + 3 * r + c];
}


// The value of lane Q of the quad, Q a constant after unrolling.
__device__ __forceinline__ double quad_lane(double v, int Q) {
    switch (Q) {
        case 0: return dpp_mov<0x00>(v);
        case 1: return dpp_mov<0x55>(v);
        case 2: return dpp_mov<0xAA>(v);
        default: return dpp_mov<0xFF>(v);
    }
}

// R rows' 32 raw panel entries eliminated against U11 (D, strictly upper triangle in LDS, zeros elsewhere) with the pivots'
// reciprocals, four lanes a row: lane q = threadIdx.x % 4 holds columns 4 m + q and ends with u(k0 + 4 m + q, row). What
// bounds it is the FP64 rate of one wavefront (a row a lane took 3.0 us), then the chain of 32 steps. Row k + 1 of U11 is
// read while row k is used.
template <int R>
__device__ __forceinline__ void eliminate_rows(double (&r)[2][kLuPanel / 4], const double (*D)[kLuPanel + 1],
                                               const double* rp) {
    constexpr int M = kLuPanel / 4;
    const int q = threadIdx.x & 3;
    double u[2][M + 1];
    auto fetch = [&](int k) {
#pragma unroll
        for (int m = k >> 2; m < M; ++m) u[k & 1][m] = D[k][4 * m + q];
        u[k & 1][M] = rp[k];
    };
    fetch(0);
#pragma unroll
    for (int k = 0; k < kLuPanel; ++k) {
        if (k + 1 < kLuPanel) fetch(k + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < R; ++e) {
            const double l = quad_lane(r[e][k >> 2], k & 3) * u[k & 1][M];
#pragma unroll
            for (int m = k >> 2; m < M; ++m) r[e][m] -= l * u[k & 1][m];  // a zero for the columns up to k
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Sums over lanes i and i ^ 32 of a (lanes 0..31) and b (lanes 32..63); over lanes i and i ^ 16 of a (even rows of 16 lanes)
// and b (odd rows).
__device__ __forceinline__ double swap32_add(double a, double b) {
    const v2u x = __builtin_bit_cast(v2u, a), y = __builtin_bit_cast(v2u, b);
    const auto lo = __builtin_amdgcn_permlane32_swap(x[0], y[0], false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(x[1], y[1], false, false);
    return __builtin_bit_cast(double, v2u{lo[0], hi[0]}) + __builtin_bit_cast(double, v2u{lo[1], hi[1]});
}
__device__ __forceinline__ double swap16_add(double a, double b) {
    const v2u x = __builtin_bit_cast(v2u, a), y = __builtin_bit_cast(v2u, b);
    const auto lo = __builtin_amdgcn_permlane16_swap(x[0], y[0], false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(x[1], y[1], false, false);
    return __builtin_bit_cast(double, v2u{lo[0], hi[0]}) + __builtin_bit_cast(double, v2u{lo[1], hi[1]});
}
// 1 / v to the last bit or its neighbour: the hardware's estimate and two Newton steps, a third of a division's chain.
__device__ __forceinline__ double reciprocal(double v) {
    double r = __builtin_amdgcn_rcp(v);
    r = fma(fma(-v, r, 1.0), r, r);
    return fma(fma(-v, r, 1.0), r, r);
}

// Elimination of an nb x nb diagonal block by one wavefront, and the block's U into the band at k0. Lane i and lane 32 + i
// hold row i's lower part (past nb the identity's): r[m] of lane half h is column 2 m + h. Column c of the block is row c of
// U: the pivot and the entries of the next one or two columns come from their lanes at once, the others through LDS (T; no
// barrier: one wavefront) a step later, so a step is the chain pivot, reciprocal, product. With all of a row in one
// lane the FP64 rate bounded it (3.4 us); with 256 threads, a barrier and a division
// a step it took 8 us.
__device__ __forceinline__ void eliminate_block_write(double* __restrict__ ab, int bw, int64_t ld, int64_t k0, int nb,
                                                      double (&r)[kLuPanel / 2], double (*T)[kLuPanel]) {
    constexpr int M = kLuPanel / 2;
    const int lane = threadIdx.x & 31, h = threadIdx.x >> 5;
    double l = 0.0, u[2][M];
#pragma unroll
    for (int c = 0; c < kLuPanel; ++c) {
        // column c is complete; l and u[(c + 1) & 1] are column c - 1, still to go into the registers from m1 on
        const v2u own = __builtin_bit_cast(v2u, r[c >> 1]);
        const auto lo = __builtin_amdgcn_permlane32_swap(own[0], own[0], false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(own[1], own[1], false, false);
        const double col = __builtin_bit_cast(double, v2u{lo[c & 1], hi[c & 1]});  // both halves: column c
        const int m0 = (c + 1) >> 1, m1 = (c >> 1) + 1;  // registers of column c + 1; first ones of the deferred c - 1
        T[c][lane] = col;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int m = m0 + 1; m < M; ++m) u[c & 1][m] = T[c][2 * m + h];
        // col / pivot with the estimate's correction off the product's chain
        const double pivot = read_lane(col, c), e0 = __builtin_amdgcn_rcp(pivot), err = fma(-pivot, e0, 1.0);
        const double q0 = col * e0, lc = fma(q0, fma(err, err, err), q0);
        if (c > 0) {
#pragma unroll
            for (int m = m1; m < M; ++m) r[m] -= l * u[(c + 1) & 1][m];
        }
        if (c + 1 < kLuPanel) {
            double next = read_lane(col, c + 1);
            if (c & 1) {  // columns c + 1 and c + 2 share the register
                const double next2 = read_lane(col, c + 2);
                next = h ? next2 : next;
            }
            r[m0] -= lc * next;
        }
        l = lc;
        __builtin_amdgcn_sched_barrier(0);
    }
    double* rows = ab + k0 * ld;
#pragma unroll 4
    for (int c = h; c < nb; c += 2)
        if (c <= lane && lane < nb && lane - c <= bw) rows[(uint32_t)(c * (int)ld + (lane - c + bw))] = T[c][lane];
}

// The first panel's diagonal block.
__global__ __launch_bounds__(64) void ldl_step_first_kernel(double* __restrict__ ab, int bw, int64_t ld, int nb) {
    __shared__ double T[kLuPanel][kLuPanel];
    const int i = threadIdx.x & 31, h = threadIdx.x >> 5;
    double r[kLuPanel / 2];
#pragma unroll
    for (int m = 0; m < kLuPanel / 2; ++m) {
        const int j = 2 * m + h;
        const bool in = i < nb && j <= i && i - j <= bw;
        const double v = ab[in ? (uint32_t)(i * (int)ld + (j - i + bw)) : 0u];
        r[m] = in ? v : i == j ? 1.0 : 0.0;
    }
    eliminate_block_write(ab, bw, ld, 0, nb, r, T);
}

// Panel [k0, k0 + 32) whose diagonal block is eliminated (U11 in the band): workgroup 0 updates and eliminates the next
// diagonal block [k1, k1 + next_nb)^2; the others take the 64 x 64 lower tiles of the trailing block
// a(i, j) -= sum_c l(i, c) u(c, j), i >= j in [k1, k1 + m), and the tiles on the diagonal write U12 of their rows.
__global__ __launch_bounds__(256) void ldl_step_kernel(double* __restrict__ ab, int bw, int64_t ld, int64_t k0,
                                                       int64_t m, int next_nb) {
    __shared__ double Ls[2 * kTile][kLuPanel + 1];  // l and u of the rows of ti, then of tj
    __shared__ double Us[kLuPanel][2 * kTile + 1];
    __shared__ double D[kLuPanel][kLuPanel + 1];
    __shared__ double rp[kLuPanel];
    const int tid = threadIdx.x;
    const int64_t k1 = k0 + kLuPanel, iend = k1 + m;
    const bool next = blockIdx.x == 0;
    int ti = 0, tj = 0;
    if (!next) {
        const int b = (int)blockIdx.x - 1;
        while ((ti + 1) * (ti + 2) / 2 <= b) ++ti;
        tj = b - ti * (ti + 1) / 2;
    } else if (next_nb <= 0) {
        return;
    }
    const int64_t i0 = k1 + (int64_t)ti * kTile, j0 = k1 + (int64_t)tj * kTile;
    const bool same = ti == tj;
    // rows of ti, and of tj where that is another tile, four lanes a row; every load goes out before the first use
    const int q4 = tid & 3, lr = tid >> 2;
    double r[2][kLuPanel / 4];
    auto load_rows = [&](double (&e)[kLuPanel / 4], int64_t first) {
        const double* raw = ab + first * ld;
        const int row = (int)(first - k1) + lr;  // within the trailing block
        const bool mine = row < (next ? next_nb : (int)m);
#pragma unroll
        for (int c4 = 0; c4 < kLuPanel / 4; ++c4) {
            const int d = row + kLuPanel - (4 * c4 + q4);  // row minus column
            const bool in = mine && d <= bw;
            const double v = raw[in ? (uint32_t)(lr * (int)ld + bw - d) : 0u];
            e[c4] = in ? v : 0.0;
        }
    };
    load_rows(r[0], i0);
    if (!same) load_rows(r[1], j0);
    double* diag = ab + k0 * ld + bw;
    double dv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = tid / kLuPanel + 8 * q, j = tid % kLuPanel;
        const bool in = j >= c && j - c <= bw;  // the pivots too
        const double v = diag[in ? (uint32_t)(c * (int)ld + j - c) : 0u];
        dv[q] = in ? v : 0.0;
    }
    const int tx = tid % 16, ty = tid / 16;
    // Entry (i, j) of the tile, and whether it is this one's to write: not the next diagonal block's
    const int di = (int)(i0 - k1), dj = (int)(j0 - k1);
    double* tile = ab + i0 * ld;
    auto place = [&](int i, int j) { return (uint32_t)(i * (int)ld + (dj + j - di - i + bw)); };
    auto writes = [&](int i, int j) {
        const int gi = di + i, gj = dj + j;
        return gi < m && gj < m && gj - gi <= bw && gi - gj <= bw && !(gi < next_nb && gj < next_nb);
    };
    double old[4][4], nv[4];
    if (next) {
        const int i = tid >> 3;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int j = (tid & 7) + 8 * q;
            const bool in = i < next_nb && j <= i && i - j <= bw;
            const double v = ab[in ? (k1 + i) * ld + (j - i + bw) : 0];
            nv[q] = in ? v : 0.0;
        }
    } else {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int bb = 0; bb < 4; ++bb) {
                const bool in = writes(ty + 16 * a, tx + 16 * bb);
                const double v = tile[in ? place(ty + 16 * a, tx + 16 * bb) : 0u];
                old[a][bb] = in ? v : 0.0;
            }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = tid / kLuPanel + 8 * q;
        const bool pivot = tid % kLuPanel == c;
        D[c][tid % kLuPanel] = pivot ? 0.0 : dv[q];
        if (pivot) rp[c] = reciprocal(dv[q]);
    }
    __syncthreads();
    auto stage = [&](const double (&e)[kLuPanel / 4], int at) {
#pragma unroll
        for (int c4 = 0; c4 < kLuPanel / 4; ++c4) {
            const int c = 4 * c4 + q4;
            Ls[at][c] = e[c4] * rp[c];
            Us[c][at] = e[c4];
        }
    };
    if (!same) {
        eliminate_rows<2>(r, D, rp);
        stage(r[0], lr);
        stage(r[1], kTile + lr);
    } else if (!next || tid < 4 * kLuPanel) {
        eliminate_rows<1>(r, D, rp);
        stage(r[0], lr);
    }
    __syncthreads();
    if (next) {
        const int i = tid >> 3;
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 16
        for (int c = 0; c < kLuPanel; ++c) {
            const double l = Ls[i][c];
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[q] += l * Us[c][(tid & 7) + 8 * q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int j = (tid & 7) + 8 * q;
            D[i][j] = i < next_nb && j <= i && i - j <= bw ? nv[q] - acc[q] : i == j ? 1.0 : 0.0;
        }
        __syncthreads();
        if (tid >= 64) return;
        double rows[kLuPanel / 2];
#pragma unroll
        for (int c2 = 0; c2 < kLuPanel / 2; ++c2) rows[c2] = D[tid & 31][2 * c2 + (tid >> 5)];
        eliminate_block_write(ab, bw, ld, k1, next_nb, rows, reinterpret_cast<double(*)[kLuPanel]>(&Ls[kTile][0]));
        return;
    }
    if (same)
        for (int e = tid; e < kLuPanel * kTile; e += 256) {
            const int c = e / kTile;
            const int64_t j = j0 + e % kTile;
            if (j < iend && j - (k0 + c) <= bw) at(ab, ld, bw, k0 + c, j) = Us[c][e % kTile];
        }
    double acc[4][4] = {};
#pragma unroll 4
    for (int c = 0; c < kLuPanel; ++c) {
        double l[4], u[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) l[a] = Ls[ty + 16 * a][c];
#pragma unroll
        for (int bb = 0; bb < 4; ++bb) u[bb] = Us[c][(same ? 0 : kTile) + tx + 16 * bb];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int bb = 0; bb < 4; ++bb) acc[a][bb] += l[a] * u[bb];
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int bb = 0; bb < 4; ++bb) {
            if (writes(ty + 16 * a, tx + 16 * bb)) tile[place(ty + 16 * a, tx + 16 * bb)] = old[a][bb] - acc[a][bb];
        }
}

// L(i, j) = U(j, i) / U(j, j) (as a product with the reciprocal) for the 64 x 64 tile of rows 64 (blockIdx.x + blockIdx.y),
// columns 64 blockIdx.x, through LDS so that both sides are contiguous.
__global__ __launch_bounds__(256) void ldl_lower_kernel(double* __restrict__ ab, int64_t n, int bw, int64_t ld) {
    __shared__ double T[kTile][kTile + 1];
    const int64_t j0 = (int64_t)blockIdx.x * kTile, i0 = j0 + (int64_t)blockIdx.y * kTile;
    for (int e = threadIdx.x; e < kTile * kTile; e += 256) {
        const int64_t j = j0 + e / kTile, i = i0 + e % kTile;
        if (i < n && j < i && i - j <= bw)
            T[e / kTile][e % kTile] = atc(ab, ld, bw, j, i) * (1.0 / atc(ab, ld, bw, j, j));
    }
    __syncthreads();
    for (int e = threadIdx.x; e < kTile * kTile; e += 256) {
        const int64_t i = i0 + e / kTile, j = j0 + e % kTile;
        if (i < n && j < i && i - j <= bw) at(ab, ld, bw, i, j) = T[e % kTile][e / kTile];
    }
}

// Inverse of the 64 x 64 diagonal block blockIdx.x of L (blockIdx.y = 0, unit lower) or U (1, upper), row-major
// at inv + (2 blockIdx.x + blockIdx.y) 64^2; rows past n padded with the identity. Lane c forms column c by
// substitution on the identity column, eight rows at a time: the sums over the rows before them are independent (one chain
// over all rows took 113 us at 3,240 DOFs).
template <bool UPPER>
__device__ __forceinline__ void block_inverse(const double* __restrict__ ab, int64_t n, int bw, int64_t ld,
                                              double* __restrict__ out, double (*T)[kTile + 2], double (*X)[kTile], double* R) {
    constexpr int G = 8;
    const int64_t r0 = (int64_t)blockIdx.x * kTile;
    const int mb = (int)min((int64_t)kTile, n - r0);
    const int c = threadIdx.x;
    const auto rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(ab) + r0 * ld, 0, (int)(mb * ld * 8), 0x00027000);
#pragma unroll 16
    for (int r = 0; r < kTile; ++r) {  // T[k][r]: the block's column k
        const bool in = r < mb && c < mb && (UPPER ? (c >= r && c - r <= bw) : (c < r && r - c <= bw));
        const v2u v = __builtin_amdgcn_raw_buffer_load_b64(rows, in ? 8 * (r * (int)ld + (c - r + bw)) : -8, 0, 0);
        T[c][r] = in ? __builtin_bit_cast(double, v) : (r == c) ? 1.0 : 0.0;
    }
    R[c] = 1.0 / T[c][c];
    __syncthreads();
    for (int g = 0; g < kTile / G; ++g) {
        const int b = UPPER ? kTile - G * (g + 1) : G * g;  // rows [b, b + G), after those already in X
        double x[G];
#pragma unroll
        for (int i = 0; i < G; ++i) x[i] = (b + i == c) ? 1.0 : 0.0;
#pragma unroll 8
        for (int m = 0; m < G * g; ++m) {
            const int k = UPPER ? kTile - 1 - m : m;
            const double xk = X[k][c];
#pragma unroll
            for (int i = 0; i < G; ++i) x[i] -= T[k][b + i] * xk;
        }
#pragma unroll
        for (int m = 0; m < G; ++m) {
            const int k = UPPER ? G - 1 - m : m;
            if (UPPER) {  // the quotient by the reciprocal and its correction
                const double t = T[b + k][b + k], rt = R[b + k], q = x[k] * rt;
                x[k] = fma(fma(-t, q, x[k]), rt, q);
            }
#pragma unroll
            for (int i = UPPER ? 0 : k + 1; i < (UPPER ? k : G); ++i) x[i] -= T[b + k][b + i] * x[k];
        }
#pragma unroll
        for (int i = 0; i < G; ++i) {
            X[b + i][c] = x[i];  // read by this lane only
            out[(b + i) * kTile + c] = x[i];
        }
    }
}
__global__ __launch_bounds__(64) void band_block_inverse_kernel(const double* __restrict__ ab, int64_t n, int bw,
                                                                int64_t ld, double* __restrict__ inv) {
    __shared__ double T[kTile][kTile + 2];
    __shared__ double X[kTile][kTile];
    __shared__ double R[kTile];
    double* out = inv + ((int64_t)blockIdx.x * 2 + blockIdx.y) * (kTile * kTile);
    if (blockIdx.y == 1) block_inverse<true>(ab, n, bw, ld, out, T, X, R);
    else block_inverse<false>(ab, n, bw, ld, out, T, X, R);
}

// x = U^-1 L^-1 b for columns [R blockIdx.x, R blockIdx.x + R) of nrhs, 256 threads. Products over a 64-entry
// tile are split by entries: wavefront g takes entries [16 g, 16 g + 16) of every row and column, and the four
// partial sums of a row block are added in wavefront order; thread (row l = tid % 64, g) then owns columns
// [g R / 4, (g + 1) R / 4) of the row. identity_first >= 0: b holds columns identity_first + j of the identity,
// whose forward solutions are zero above row identity_first + j; the forward pass starts at the row block of the
// first column (rows above it written zero). x may alias b.
template <int R>
__global__ __launch_bounds__(256) void band_solve_blocked_kernel(const double* __restrict__ ab,
                                                                 const double* __restrict__ inv, int64_t n, int bw,
                                                                 int64_t ld, int nrhs, const double* b, int64_t ldb,
                                                                 double* x, int64_t ldx, int64_t identity_first) {
    constexpr int CPT = R / 4;               // columns each thread finishes
    constexpr int PA = kTile * kTile / 256;  // tile values each thread stages
    constexpr int PY = kTile * R / 256;
    constexpr int KW = kTile / 4;            // tile entries per wavefront
    static_assert(4 * R * kTile <= kTile * (kTile + 1), "partial sums fit in At");
    __shared__ double At[kTile][kTile + 1];  // At[k][row]; also the wavefronts' partial sums
    __shared__ double Ys[kTile][R + 2];      // Ys[k][column] (rows 16-byte aligned)
    __shared__ double Rs[kTile][R + 2];      // Rs[row][column]
    const int tid = threadIdx.x, l = tid & 63, g = tid >> 6, kk0 = tid & 63;
    const int64_t j0 = (int64_t)blockIdx.x * R;
    const int64_t nblk = (n + kTile - 1) / kTile;
    int64_t sb = 0;
    if (identity_first >= 0) {
        sb = (identity_first + j0) / kTile;
        const int64_t rows = sb * kTile;
        for (int64_t e = tid; e < rows * R; e += 256) {
            const int64_t cc = e / rows, i = e - cc * rows;
            if (j0 + cc < nrhs) x[(j0 + cc) * ldx + i] = 0.0;
        }
    }
    double pa[PA], py[PY];
    // Tile [kt, kt + kn) of row block r0 into registers (thread: entry kk0, rows g + 4 q; columns g + 4 q of x),
    // loads issued unconditionally from clamped addresses. The forward pass reads L (k < i), the backward U (k > i).
    auto load_tile = [&](int64_t r0, int64_t rend, int64_t kt, int kn, bool lower) {
        const int64_t k = kt + kk0;
#pragma unroll
        for (int q = 0; q < PA; ++q) {
            const int64_t i = r0 + g + 4 * q;
            const bool in = kk0 < kn && i < rend && (lower ? i - k <= bw : k - i <= bw);
            const double v = ab[in ? i * ld + (k - i + bw) : 0];
            pa[q] = in ? v : 0.0;
        }
#pragma unroll
        for (int q = 0; q < PY; ++q) {
            const int64_t j = j0 + g + 4 * q;
            const bool in = kk0 < kn && j < nrhs;
            const double v = x[in ? j * ldx + k : 0];
            py[q] = in ? v : 0.0;
        }
    };
    auto store_tile = [&]() {
#pragma unroll
        for (int q = 0; q < PA; ++q) At[kk0][g + 4 * q] = pa[q];
#pragma unroll
        for (int q = 0; q < PY; ++q) Ys[kk0][g + 4 * q] = py[q];
    };
    // acc[c] += sum over this wavefront's entries of At[k][l] S[k][c]
    auto kpart = [&](const double (*S)[R + 2], double* acc) {
#pragma unroll
        for (int u = 0; u < KW; ++u) {
            const int kk = g * KW + u;
            const double a = At[kk][l];
#pragma unroll
            for (int c = 0; c < R; ++c) acc[c] += a * S[kk][c];
        }
    };
    // out[q] = the four wavefronts' partials of column g CPT + q of row l, added in wavefront order. At must be
    // free on entry; it is free again on return.
    auto reduce = [&](const double* acc, double* out) {
        double* P = &At[0][0];
#pragma unroll
        for (int c = 0; c < R; ++c) P[(g * R + c) * kTile + l] = acc[c];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            const int c = g * CPT + q;
            out[q] = ((P[c * kTile + l] + P[(R + c) * kTile + l]) + P[(2 * R + c) * kTile + l]) +
                     P[(3 * R + c) * kTile + l];
        }
        __syncthreads();
    };
    // tot = the row block's band products with the solved entries [kbeg, kend); At free on return
    auto products = [&](int64_t r0, int64_t rend, int64_t kbeg, int64_t kend, bool lower, double* tot) {
        double acc[R];
#pragma unroll
        for (int c = 0; c < R; ++c) acc[c] = 0.0;
        if (kbeg < kend) {
            load_tile(r0, rend, kbeg, (int)min((int64_t)kTile, kend - kbeg), lower);
            for (int64_t kt = kbeg; kt < kend; kt += kTile) {
                __syncthreads();  // the last tile's readers are done
                store_tile();
                __syncthreads();
                const int64_t kn = kt + kTile;
                if (kn < kend) load_tile(r0, rend, kn, (int)min((int64_t)kTile, kend - kn), lower);
                kpart(Ys, acc);
            }
            __syncthreads();
        }
        reduce(acc, tot);
    };
    // x rows [r0, rend) of the block's columns = inverse block (row-major at blk) times Rs
    auto triangle = [&](const double* __restrict__ blk, int64_t r0, int64_t rend) {
#pragma unroll
        for (int q = 0; q < PA; ++q) At[kk0][g + 4 * q] = blk[(g + 4 * q) * kTile + kk0];
        __syncthreads();  // At and Rs complete
        double acc[R];
#pragma unroll
        for (int c = 0; c < R; ++c) acc[c] = 0.0;
        kpart(Rs, acc);
        __syncthreads();
        double y[CPT];
        reduce(acc, y);
        const int64_t i = r0 + l;
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            const int64_t j = j0 + g * CPT + q;
            if (i < rend && j < nrhs) x[j * ldx + i] = y[q];
        }
        __syncthreads();  // x rows written before the next block reads them
    };
    double tot[CPT];
    for (int64_t rb = sb; rb < nblk; ++rb) {  // forward: y = L^-1 b
        const int64_t r0 = rb * kTile;
        products(r0, n, std::max(sb * kTile, r0 - bw), r0, true, tot);
        const int64_t i = r0 + l;
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            const int64_t j = j0 + g * CPT + q;
            Rs[l][g * CPT + q] = (i < n && j < nrhs) ? b[j * ldb + i] - tot[q] : 0.0;
        }
        triangle(inv + rb * 2 * (kTile * kTile), r0, n);
    }
    for (int64_t rb = nblk - 1; rb >= 0; --rb) {  // backward: x = U^-1 y
        const int64_t r0 = rb * kTile, r1 = std::min(n, r0 + kTile);
        products(r0, r1, r1, std::min(n, r1 + bw), false, tot);
        const int64_t i = r0 + l;
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            const int64_t j = j0 + g * CPT + q;
            Rs[l][g * CPT + q] = (i < r1 && j < nrhs) ? x[j * ldx + i] - tot[q] : 0.0;
        }
        triangle(inv + (rb * 2 + 1) * (kTile * kTile), r0, r1);
    }
}

// x = U^-1 L^-1 b for one column per workgroup of 1,024 threads, x in LDS, bandwidth up to 64 S. Each wavefront takes four
// rows of a 64-row block, its lanes along the band (512 contiguous bytes, one read of x for the four rows): their band
// products with the entries solved before, then the block's triangle as a product with its inverse, sixteen lanes a row.
// The next block's band entries and inverse are on their way meanwhile: nothing that is read depends on x. What bounds it
// is the one compute unit's load rate. The tiled kernel above staged 6 tiles a block through LDS one after another, 14 us
// a block at bandwidth 356.
template <int S>
__global__ __launch_bounds__(1024) void band_solve_column_kernel(const double* __restrict__ ab,
                                                                 const double* __restrict__ inv, int64_t n, int bw,
                                                                 int64_t ld, const double* b, int64_t ldb, double* x,
                                                                 int64_t ldx) {
    extern __shared__ double lds[];  // 64 S zeros, x, kTile + 64 S zeros
    __shared__ double rs[kTile];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, r = t >> 4, q = t & 15;
    const int nblk = (int)((n + kTile - 1) / kTile);
    double* xs = lds + 64 * S;
    for (int i = t - 64 * S; i < (int)n + kTile + 64 * S; i += 1024)
        xs[i] = i >= 0 && i < n ? b[blockIdx.x * ldb + i] : 0.0;
    double a[4][S], v[4];
    // Entries e = lane + 64 s of row r0 + 4 w + k outside its block: columns r0 - 1 - e (lower) or r0 + 64 + e. Those past the
    // row's last one are zero.
    auto load = [&](int rb, bool lower, int s) {
        const int r0 = rb * kTile;
        const auto rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(ab) + (int64_t)r0 * ld, 0,
                                                            (int)(min((int64_t)kTile, n - r0) * ld * 8), 0x00027000);
        int e = lane + 64 * s;
        asm volatile("" : "+v"(e));  // else all positions stay in registers
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int row = 4 * w + k;
            const int emax = r0 + row >= n ? -1 : lower ? min(bw - 1 - row, r0 - 1) : min(bw - kTile + row, (int)n - 1 - r0 - kTile);
            const int at = 8 * (row * (int)ld + bw + (lower ? -1 - row - e : kTile - row + e));
            a[k][s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rows, e <= emax ? at : -8, 0, 0));
        }
    };
    auto load_inverse = [&](int rb, bool lower) {
        const double* blk = inv + (int64_t)(2 * rb + (lower ? 0 : 1)) * (kTile * kTile);
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = blk[(uint32_t)(r * kTile + 4 * q + c)];
    };
    auto solve = [&](int rb, bool lower, int next, bool next_lower) {
        const int r0 = rb * kTile, i = r0 + r;
        const double* xe = xs + (lower ? r0 - 1 - lane : r0 + kTile + lane);
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const double xv = xe[lower ? -64 * s : 64 * s];
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[k] += a[k][s] * xv;
            __builtin_amdgcn_sched_barrier(0);
            load(next, next_lower, s);
            __builtin_amdgcn_sched_barrier(0);
        }
        // four sums over 64 lanes: the 16 lanes of row r end with its sum
        const double sum = group_sum<16>(swap16_add(swap32_add(acc[0], acc[2]), swap32_add(acc[1], acc[3])));
        if (q == 0) rs[r] = i < n ? xs[i] - sum : 0.0;
        __syncthreads();
        double y = 0.0;
#pragma unroll
        for (int c = 0; c < 4; ++c) y += v[c] * rs[4 * q + c];
        load_inverse(next, next_lower);
        y = group_sum<16>(y);
        if (q == 0 && i < n) xs[i] = y;
        __syncthreads();
    };
#pragma unroll
    for (int s = 0; s < S; ++s) load(0, true, s);
    load_inverse(0, true);
    __syncthreads();
    for (int rb = 0; rb + 1 < nblk; ++rb) solve(rb, true, rb + 1, true);
    solve(nblk - 1, true, nblk - 1, false);
    for (int rb = nblk - 1; rb >= 0; --rb) solve(rb, false, max(rb - 1, 0), false);
    for (int64_t i = t; i < n; i += 1024) x[blockIdx.x * ldx + i] = xs[i];
}
constexpr int kColumnMaxBw = 512;       // 8 entries of a row a lane: 124 of the 128 registers
constexpr int64_t kColumnMaxN = 18000;  // x and its margins within 153 KB of LDS

template <int S>
void solve_columns(const DeviceBandLU& lu, int nrhs, const double* b, int64_t ldb, double* x, int64_t ldx, hipStream_t s) {
    launch_k((band_solve_column_kernel<S>), dim3(nrhs), dim3(1024), (uint32_t)((lu.n + 128 * S + kTile) * sizeof(double)), s,
             (const double*)lu.ab, (const double*)lu.inv, lu.n, lu.bw, lu.ld, b, ldb, x, ldx);
}

__global__ __launch_bounds__(256) void identity_columns_kernel(int64_t n, int64_t first, int count,
                                                               double* __restrict__ out) {
    const int64_t total = n * (int64_t)count;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = t / n, i = t - j * n;
        out[t] = (i == first + j) ? 1.0 : 0.0;
    }
}

__global__ __launch_bounds__(256) void zero_bc_rows_cols_kernel(int64_t n, int64_t first, int count,
                                                                const uint8_t* __restrict__ mask,
                                                                double* __restrict__ out) {
    const int64_t total = n * (int64_t)count;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = t / n, i = t - j * n;
        if (mask[i] || mask[first + j]) out[t] = 0.0;
    }
}

__global__ __launch_bounds__(256) void zero_masked_rows_kernel(int64_t n, int count, const uint8_t* __restrict__ mask,
                                                               double* __restrict__ x) {
    const int64_t total = n * (int64_t)count;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x)
        if (mask[t % n]) x[t] = 0.0;
}

unsigned grid_for(int64_t count, int per) {
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>((count + per - 1) / per, 65536));
}

}  // namespace

int64_t band_blocks(int64_t n) { return (n + kTile - 1) / kTile; }

size_t band_bytes(int64_t n, int bw) {
    return ((size_t)n * (size_t)(2 * bw + 1) + (size_t)band_blocks(n) * 2 * kTile * kTile) * sizeof(double);
}

void launch_band_fill(DeviceBandLU& lu, int64_t num_blocks, const int* blk_row, const int* colidx, const double* S,
                      hipStream_t s) {
    const int64_t count = lu.n * lu.ld;
    launch_k(band_zero_kernel, dim3(grid_for(count, 256)), dim3(256), 0, s, lu.ab, count);
    if (num_blocks > 0)
        launch_k(band_fill_kernel, dim3((unsigned)((num_blocks + 255) / 256)), dim3(256), 0, s, lu.ab, lu.ld, lu.bw,
                 num_blocks, blk_row, colidx, S);
}

void launch_band_factor(DeviceBandLU& lu, hipStream_t s) {
    if (lu.n <= 0) return;
    if (!lu.inv) throw std::runtime_error("band LU without block-inverse storage");
    launch_k(ldl_step_first_kernel, dim3(1), dim3(64), 0, s, lu.ab, lu.bw, lu.ld, (int)std::min<int64_t>(lu.n, kLuPanel));
    for (int64_t k1 = kLuPanel; k1 < lu.n; k1 += kLuPanel) {
        const int64_t m = std::min(lu.n, k1 + lu.bw) - k1, tiles = (m + kTile - 1) / kTile;
        launch_k(ldl_step_kernel, dim3((unsigned)(1 + tiles * (tiles + 1) / 2)), dim3(256), 0, s, lu.ab, lu.bw, lu.ld,
                 k1 - kLuPanel, m, (int)std::min<int64_t>(kLuPanel, lu.n - k1));
    }
    launch_k(ldl_lower_kernel, dim3((unsigned)band_blocks(lu.n), (unsigned)((lu.bw + kTile - 1) / kTile + 1)), dim3(256),
             0, s, lu.ab, lu.n, lu.bw, lu.ld);
    launch_k(band_block_inverse_kernel, dim3((unsigned)band_blocks(lu.n), 2), dim3(64), 0, s, (const double*)lu.ab,
             lu.n, lu.bw, lu.ld, lu.inv);
}

void launch_band_solve(const DeviceBandLU& lu, int nrhs, const double* b, int64_t ldb, double* x, int64_t ldx,
                       hipStream_t s, int64_t identity_first, int64_t total) {
    if (nrhs <= 0 || lu.n == 0) return;
    // A workgroup per column: 1 column 0.32 ms against 1.43 with the tiled kernel at 3,240 DOFs, bandwidth 356; 64 columns
    // 0.52 against 2.53 (0.26 and 0.57 at 1,488 x 77, 0.88 and 4.9 at 5,184 x 470); 512 in one launch 1.9 against 4.1 (1.3 and
    // 2.3, 2.5 and 6.4). Two more rounds of 256 workgroups would bring the two level near 1,000. The line is drawn by the
    // whole request (total): every entry point passes it on, so that the results do not depend on how one cuts the request.
    // Columns of the identity stay with the tiled kernel, which skips the rows above them.
    if (std::max<int64_t>(nrhs, total) <= kColumnSolves && identity_first < 0 && lu.bw <= kColumnMaxBw && lu.n <= kColumnMaxN) {
        if (lu.bw <= 128) return solve_columns<2>(lu, nrhs, b, ldb, x, ldx, s);
        if (lu.bw <= 256) return solve_columns<4>(lu, nrhs, b, ldb, x, ldx, s);
        if (lu.bw <= 384) return solve_columns<6>(lu, nrhs, b, ldb, x, ldx, s);
        return solve_columns<8>(lu, nrhs, b, ldb, x, ldx, s);
    }
    if (nrhs >= 64)
        launch_k(band_solve_blocked_kernel<16>, dim3((unsigned)((nrhs + 15) / 16)), dim3(256), 0, s,
                 (const double*)lu.ab, (const double*)lu.inv, lu.n, lu.bw, lu.ld, nrhs, b, ldb, x, ldx,
                 identity_first);
    else
        launch_k(band_solve_blocked_kernel<4>, dim3((unsigned)((nrhs + 3) / 4)), dim3(256), 0, s,
                 (const double*)lu.ab, (const double*)lu.inv, lu.n, lu.bw, lu.ld, nrhs, b, ldb, x, ldx,
                 identity_first);
}

void launch_identity_columns(int64_t n, int64_t first, int count, double* out, hipStream_t s) {
    launch_k(identity_columns_kernel, dim3(grid_for(n * (int64_t)count, 256)), dim3(256), 0, s, n, first, count, out);
}

void launch_zero_bc_rows_cols(int64_t n, int64_t first, int count, const uint8_t* mask, double* out, hipStream_t s) {
    launch_k(zero_bc_rows_cols_kernel, dim3(grid_for(n * (int64_t)count, 256)), dim3(256), 0, s, n, first, count, mask,
             out);
}

// Partial products of a dense column-major C: workgroup (row tile, column chunk), one thread per row, the
// chunk's columns in order; the chunk's x values staged in LDS.
__global__ __launch_bounds__(256) void dense_gemv_part_kernel(int64_t n, const double* __restrict__ C,
                                                              const double* __restrict__ x,
                                                              double* __restrict__ part) {
    __shared__ double xs[kGemvCols];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t j0 = (int64_t)blockIdx.y * kGemvCols;
    const int64_t j1 = min(n, j0 + kGemvCols);
    if (threadIdx.x < kGemvCols && j0 + threadIdx.x < j1) xs[threadIdx.x] = x[j0 + threadIdx.x];
    __syncthreads();
    if (i >= n) return;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    const double* col = C + j0 * n + i;
    const int m = (int)(j1 - j0);
    int k = 0;
    for (; k + 3 < m; k += 4) {
        a0 += col[(int64_t)k * n] * xs[k];
        a1 += col[(int64_t)(k + 1) * n] * xs[k + 1];
        a2 += col[(int64_t)(k + 2) * n] * xs[k + 2];
        a3 += col[(int64_t)(k + 3) * n] * xs[k + 3];
    }
    for (; k < m; ++k) a0 += col[(int64_t)k * n] * xs[k];
    part[(int64_t)blockIdx.y * n + i] = (a0 + a1) + (a2 + a3);
}

// y[i] = the chunks' partials of row i added in chunk order; 64 rows per workgroup, loads 8 chunks at a time.
__global__ __launch_bounds__(64) void dense_gemv_sum_kernel(int64_t n, int64_t chunks,
                                                            const double* __restrict__ part, double* __restrict__ y) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double acc = 0.0;
    int64_t c = 0;
    for (; c + 8 <= chunks; c += 8) {
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = part[(c + q) * n + i];
#pragma unroll
        for (int q = 0; q < 8; ++q) acc += v[q];
    }
    for (; c < chunks; ++c) acc += part[c * n + i];
    y[i] = acc;
}

void launch_dense_gemv(int64_t n, const double* C, const double* x, double* part, double* y, hipStream_t s) {
    if (n <= 0) return;
    if (n > (int64_t)65536 * 64) throw std::runtime_error("dense GEMV: more rows than one grid covers");
    const int64_t chunks = gemv_chunks(n);
    launch_k(dense_gemv_part_kernel, dim3(grid_for(n, 256), (unsigned)chunks), dim3(256), 0, s, n, C, x, part);
    launch_k(dense_gemv_sum_kernel, dim3(grid_for(n, 64)), dim3(64), 0, s, n, chunks, (const double*)part, y);
}

void launch_zero_masked_rows(int64_t n, int count, const uint8_t* mask, double* x, hipStream_t s) {
    launch_k(zero_masked_rows_kernel, dim3(grid_for(n * (int64_t)count, 256)), dim3(256), 0, s, n, count, mask, x);
}

}  // namespace femgpu
