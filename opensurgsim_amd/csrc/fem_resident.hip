// Conjugate gradients with the operator held on the chip (see fem_resident.hpp).
//
// The recurrence is the one-kernel iteration's (fem_kernels.hip): Eigen's ConjugateGradient
// (Math/LinearSparseSolveAndInverse.cpp:99-129 over Eigen 3.3's conjugate_gradient) with the next |r|^2 and r.z
// expanded from seven sums of the iteration before, so that an iteration needs one exchange between workgroups.
// Here one launch runs every iteration: 256 CUs hold 512 KB of registers and 160 KB of LDS each, which takes the
// whole operator of a mesh of some 60,000 to 100,000 nodes. A launch per iteration streams it from the
// Infinity Cache or HBM every time and pays the dispatch and the chain at its start.
//
// Workgroup g owns a compact set of block rows (a k-d partition of the nodes, so that few columns lie outside it).
//   - A lane keeps up to nb blocks of one block row in registers; a row takes ceil(degree / nb) lanes.
//   - p of every column the workgroup touches is in LDS; z of its halo columns too, so that only w = D q of the
//     halo columns crosses workgroups: z -= alpha w and p = z + beta p are repeated by every workgroup that
//     needs the column, with the owner's arithmetic.
//   - r, x, q, w of its own rows stay in LDS.
// Exchange between workgroups: a workgroup stores w of its rows and its seven sums as 64-bit words that are both the value
// and the notice that it is there, so that no store has to wait for another one. Stores write through to the point of
// coherence and polls bypass the caches that are not coherent across XCDs (agent scope).
//   - Sums: eight words a workgroup (64 bytes, one store), kResEmpty until the sum arrives. Every workgroup polls those of all.
//     They are kept apart for four iterations: in iteration k a workgroup empties its words of iteration k - 2 for k + 2.
//     Nobody reads those any more: this workgroup has seen the sums of k - 1 of every workgroup, each stored after that
//     one had seen k - 2. Nobody polls them too early: a workgroup polls k + 2 after it has seen this one's sums of k + 1,
//     stored after this wave has waited for its stores of iteration k (vmcnt(0) in the poll).
//   - w: words of 32 bits of value and the iteration + 1 as a tag; a workgroup polls the rows of its halo. w is
//     double-buffered by parity: w of k + 1 replaces that of k - 1 after the writer has seen the sums of k of every
//     workgroup, each stored after that one had used its halo's w of k - 1.
// At the end every workgroup leaves at the same iteration k, which needs the sums of k - 1 but not its halo: it clears the
// tags of its rows for the next launch. The sums are emptied by the solve's start.
// Every wait is bounded (ResidentArgs::wait_ticks): the launch does not rely on all of its workgroups being
// resident at once. A workgroup that gives up marks the solve (CgScalars::pad) and leaves x alone; the others see
// the mark and leave too, and the host clears everything and solves with one launch per iteration instead.
#include "fem_resident.hpp"
#include "fem_reduce.hpp"

#include <algorithm>
#include <array>
#include <atomic>
#include <future>
#include <numeric>
#include <stdexcept>
#include <thread>

namespace femgpu {

namespace {

constexpr long long kResMarkTicks = 2000;  // a wait of 20 us looks at the others' mark

template <typename T>
__device__ __forceinline__ void put(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T get(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The two halves of a double exchanged between register pairs by v_permlane{32,16}_swap: a keeps its lanes 0-31
// (rows 0 and 2 of 16) and takes b's in the others' place; b takes a's.
__device__ __forceinline__ void swap32(double& a, double& b) {
    const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    a = __builtin_bit_cast(double, (uint64_t)hi[0] << 32 | lo[0]);
    b = __builtin_bit_cast(double, (uint64_t)hi[1] << 32 | lo[1]);
}
__device__ __forceinline__ void swap16(double& a, double& b) {
    const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    a = __builtin_bit_cast(double, (uint64_t)hi[0] << 32 | lo[0]);
    b = __builtin_bit_cast(double, (uint64_t)hi[1] << 32 | lo[1]);
}
// Wave totals of eight values: lane 16 q of the wave ends with the totals of v[2 q] (first) and v[2 q + 1] (second). Two
// exchange steps halve the registers, so it takes a third of the instructions of eight separate butterflies.
__device__ __forceinline__ void wave_totals8(const double (&v)[8], double& first, double& second) {
    double r[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // lanes 0-31: v[j], lanes 32-63: v[j + 4]
        double a = v[j], b = v[j + 4];
        swap32(a, b);
        r[j] = a + b;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {  // rows of 16 lanes: v[j], v[j + 2], v[j + 4], v[j + 6]
        swap16(r[j], r[j + 2]);
        r[j] += r[j + 2];
    }
    first = group_sum<16>(r[0]);
    second = group_sum<16>(r[1]);
}
// Sum over the lanes of the wave with the same lane % 8, in every lane.
__device__ __forceinline__ double sum_mod8(double v) {
    v += dpp_mov<0x128>(v);  // row_ror:8
    double b = v;
    swap16(v, b);
    v += b;
    b = v;
    swap32(v, b);
    return v + b;
}

// A row's w as tagged words, 24 (float) or 48 bytes, moved 16 bytes at a time. Every 64-bit word speaks for itself, so it
// does not matter whether a wider access is seen whole.
constexpr int kAgentScope = 1 << 4;  // sc1: past the caches that are not coherent across XCDs
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
template <typename TV>
constexpr int kRowBytes = 6 * sizeof(TV);
template <typename TV>
struct TaggedRow {
    static constexpr int kWords = 3 * sizeof(TV) / 4;
    unsigned v[kWords], tag[kWords];
    __device__ __forceinline__ bool is(unsigned t) const {
        bool all = true;
#pragma unroll
        for (int i = 0; i < kWords; ++i) all &= tag[i] == t;
        return all;
    }
    __device__ __forceinline__ TV get(int c) const {
        if constexpr (sizeof(TV) == 4) return __builtin_bit_cast(float, v[c]);
        else return __builtin_bit_cast(double, (uint64_t)v[2 * c + 1] << 32 | v[2 * c]);
    }
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rows, int row) {
#pragma unroll
        for (int i = 0; i < kWords / 2; ++i) {
            const v4u d = __builtin_amdgcn_raw_buffer_load_b128(rows, kRowBytes<TV> * row + 16 * i, 0, kAgentScope);
            v[2 * i] = d[0];
            tag[2 * i] = d[1];
            v[2 * i + 1] = d[2];
            tag[2 * i + 1] = d[3];
        }
        if constexpr (kWords % 2 != 0) {
            const v2u d = __builtin_amdgcn_raw_buffer_load_b64(rows, kRowBytes<TV> * row + 8 * (kWords - 1), 0, kAgentScope);
            v[kWords - 1] = d[0];
            tag[kWords - 1] = d[1];
        }
    }
};
template <typename TV>
__device__ __forceinline__ void put_row(__amdgpu_buffer_rsrc_t rows, int row, const TV (&w)[3], unsigned tag) {
    unsigned v[6];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if constexpr (sizeof(TV) == 4) v[c] = __builtin_bit_cast(unsigned, w[c]);
        else {
            v[2 * c] = (unsigned)__builtin_bit_cast(uint64_t, w[c]);
            v[2 * c + 1] = (unsigned)(__builtin_bit_cast(uint64_t, w[c]) >> 32);
        }
    }
    constexpr int kWords = TaggedRow<TV>::kWords;
#pragma unroll
    for (int i = 0; i < kWords / 2; ++i)
        __builtin_amdgcn_raw_buffer_store_b128(v4u{v[2 * i], tag, v[2 * i + 1], tag}, rows, kRowBytes<TV> * row + 16 * i, 0,
                                               kAgentScope);
    if constexpr (kWords % 2 != 0)
        __builtin_amdgcn_raw_buffer_store_b64(v2u{v[kWords - 1], tag}, rows, kRowBytes<TV> * row + 8 * (kWords - 1), 0,
                                              kAgentScope);
}
__device__ __forceinline__ unsigned long long sum_word(double s) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, s);
    return u == kResEmpty ? 0x7ff8000000000000ull : u;  // a NaN with the empty word's payload
}

// Whether x, r, q, w, z and the preconditioner of the own row and z of the halo stay in registers beside the blocks;
// otherwise they are in LDS.
template <typename TV, int NB>
constexpr bool own_in_registers() {
    return 9 * NB * (int)sizeof(TV) / 4 <= 100;
}
// Dynamic LDS (values): p of the columns and one zero column, the lanes' row parts, and the own rows' vectors where they
// are not in registers.
constexpr int kResMaxCols = 3 * kResThreads;  // own rows and halo columns; the next one is the zero column
constexpr int lds_part() { return 3 * (kResMaxCols + 1) + 1; }
template <typename TV, int NB>
constexpr size_t lds_bytes() {
    return (lds_part() + (size_t)(own_in_registers<TV, NB>() ? 6 : 3 + 15 + 6 + (sizeof(TV) == 4 ? 9 : 3)) * kResThreads) *
           sizeof(TV);
}

// N values of this thread, in registers or in LDS at a constant place.
template <typename TV, int N, bool REGS>
struct Own;
template <typename TV, int N>
struct Own<TV, N, true> {
    TV v[N];
    __device__ __forceinline__ Own(TV*, int) {}
    __device__ __forceinline__ TV get(int, int c) const { return v[c]; }
    __device__ __forceinline__ void set(int, int c, TV x) { v[c] = x; }
};
template <typename TV, int N>
struct Own<TV, N, false> {
    TV* p;
    __device__ __forceinline__ Own(TV* lds, int slot) : p(lds + slot * kResThreads) {}
    __device__ __forceinline__ TV get(int t, int c) const { return p[c * kResThreads + t]; }
    __device__ __forceinline__ void set(int t, int c, TV x) { p[c * kResThreads + t] = x; }
};

template <typename TV, int NB>
__global__ __launch_bounds__(kResThreads, 2) void cg_resident_kernel(ResidentArgs a) {
    constexpr bool kBlockPc = sizeof(TV) == 4, kRegs = own_in_registers<TV, NB>();
    constexpr int kWaves = kResThreads / 64, kPc = kBlockPc ? 9 : 3;
    extern __shared__ double res_lds[];
    __shared__ double wsum[kWaves * kResWords], rsum[kWaves * kResWords];
    __shared__ int gave_up;
    int4 wg;  // first workgroup of its solve, workgroups, group, solve
    if (a.t.wg) {
        wg = a.t.wg[blockIdx.x];
    } else {
        const int solve = blockIdx.x / a.t.groups;
        wg = make_int4(solve * a.t.groups, a.t.groups, (int)blockIdx.x - solve * a.t.groups, solve);
    }
    CgScalars* const sc = a.sc + wg.w;
    if (sc->done) return;  // by the solve's start, the same for every workgroup
    const int g = wg.z, G = wg.y;
    const int max_iter = a.max_iters ? a.max_iters[wg.w] : a.max_iter;
    const TV* const r_start = (const TV*)a.r + wg.w * a.stride;
    const TV* const z_start = (const TV*)a.z + wg.w * a.stride;
    TV* const x_out = (TV*)a.x + wg.w * a.stride;
    int t = threadIdx.x;
    const int4 info = a.t.group[g];
    const int row0 = info.x, nrows = info.y, halo0 = info.z, nhalo = info.w;
    TV* lds = (TV*)res_lds;
    TV* P = lds;
    TV* part = lds + lds_part();
    Own<TV, 3, kRegs> X(part, 3), R(part, 6), Q(part, 9), Wv(part, 12), Z(part, 15);
    Own<TV, 3, kRegs> ZH(part, 18);
    Own<TV, 3, false> ZF(part, kRegs ? 3 : 21);  // halo columns beyond the first 512
    Own<TV, kPc, kRegs> D(part, 24);
    TV po[3] = {0, 0, 0}, ph[3] = {0, 0, 0};  // kRegs: p of the own row and of halo column t, as in P
    auto own_p = [&](int t, int c) { return kRegs ? po[c] : t < nrows ? P[3 * t + c] : TV(0); };
    // without a row: zeros, so that the row's part of an iteration needs no branch
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        X.set(t, c, TV(0));
        R.set(t, c, TV(0));
        Z.set(t, c, TV(0));
        Q.set(t, c, TV(0));
        Wv.set(t, c, TV(0));
    }
#pragma unroll
    for (int c = 0; c < kPc; ++c) D.set(t, c, TV(0));

    // this lane's blocks
    TV m[NB][9];
    uint32_t cpk[(NB + 1) / 2];  // byte offsets of the local columns in P, two to a register
    int pi;                      // where this lane's part of its row goes: a row's parts side by side
    {
        const int64_t li = (int64_t)g * kResThreads + t;
        const int cnt = a.t.lane_info[li] & 0xff;
        pi = 3 * (a.t.lane_info[li] >> 8);
        const TV* S = (const TV*)a.S + 9 * (int64_t)a.t.lane_k0[li];
        // every lane loads nb blocks (its last one again, the operator's first one where it has none), so that no load waits on
        // a branch
#pragma unroll
        for (int s = 0; s < NB; ++s) {
            const TV* B = S + 9 * (s < cnt ? s : max(cnt - 1, 0));
#pragma unroll
            for (int i = 0; i < 9; ++i) m[s][i] = B[i];
        }
#pragma unroll
        for (int s = 0; s < NB; ++s)
#pragma unroll
            for (int i = 0; i < 9; ++i) m[s][i] = s < cnt ? m[s][i] : TV(0);
        const uint16_t* cl = a.t.cols + (int64_t)g * NB * kResThreads + t;
#pragma unroll
        for (int s = 0; s < NB; s += 2)
            cpk[s / 2] = cl[(int64_t)s * kResThreads] |
                         (s + 1 < NB ? (uint32_t)cl[(int64_t)(s + 1) * kResThreads] << 16 : 0u);
    }
    // this thread's row (t < nrows), its halo columns t, t + 512 and the columns' start
    int l01 = 0, node = 0, hp[2] = {0, 0};
    if (t < nrows) {
        const uint16_t* rl = a.t.row_lane + (int64_t)g * (kResThreads + 1) + t;
        l01 = rl[0] | rl[1] << 16;
        node = a.t.row_node[row0 + t];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const TV z = z_start[3 * (int64_t)node + c];
            Z.set(t, c, z);
            P[3 * t + c] = z;
            po[c] = z;
            X.set(t, c, x_out[3 * (int64_t)node + c]);
            R.set(t, c, r_start[3 * (int64_t)node + c]);
        }
#pragma unroll
        for (int c = 0; c < kPc; ++c) D.set(t, c, ((const TV*)a.dinv)[kPc * (int64_t)node + c]);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int h = t + kResThreads * q;
        if (h < nhalo) {
            hp[q] = a.t.halo_pos[halo0 + h];
            const int64_t hn = a.t.halo_node[halo0 + h];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const TV z = z_start[3 * hn + c];
                if (q == 0) {
                    ZH.set(t, c, z);
                    ph[c] = z;
                } else {
                    ZF.set(t, c, z);
                }
                P[3 * (nrows + h) + c] = z;
            }
        }
    }
    if (t < 3) P[3 * kResMaxCols + t] = TV(0);
    if (t == 0) gave_up = 0;
    const double threshold = sc->threshold;
    const int rows = a.t.rows;
    const auto ring = [&](int k) {  // w of iteration k
        return __builtin_amdgcn_make_buffer_rsrc((char*)a.exch + ((int64_t)wg.w * (a.stride ? 2 : 0) + (k & 1)) * rows * kRowBytes<TV>, 0,
                                                 rows * kRowBytes<TV>, 0x00020000);
    };
    __syncthreads();

    for (int k = 0;; ++k) {
        asm volatile("" : "+v"(t));  // addresses are formed anew instead of holding registers through the loop
        const int wave = t >> 6, lane = t & 63;
        if (k > 0) {
            // the sums of iteration k - 1: thread t takes words t, t + 512, ... (component t & 7); its halo's w with them
            const unsigned long long* words = a.slots + (((k - 1) & (kResRing - 1)) * kResMaxGroups + wg.x) * kResWords + t;
            const auto ex = ring(k - 1);
            constexpr int kPer = kResMaxGroups * kResWords / kResThreads;
            unsigned long long u[kPer];
#pragma unroll
            for (int q = 0; q < kPer; ++q) u[q] = t + kResThreads * q < kResWords * G ? kResEmpty : 0ull;
            const long long t0 = wall_clock64();
            auto too_long = [&]() {
                const long long dt = wall_clock64() - t0;
                return dt > a.wait_ticks || (dt > kResMarkTicks && get(&sc->pad) != 0);
            };
            for (;;) {  // asks again for what has not arrived
#pragma unroll
                for (int q = 0; q < kPer; ++q)
                    if (u[q] == kResEmpty) u[q] = get(&words[kResThreads * q]);
                bool empty = false;
#pragma unroll
                for (int q = 0; q < kPer; ++q) empty |= u[q] == kResEmpty;
                if (!__any(empty)) break;
                if (too_long()) {
                    put(&sc->pad, 1);
                    gave_up = 1;
                    break;
                }
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the words emptied in iteration k - 1 are empty
            // the halo's w of iteration k - 1, on its way while the sums are added up
            TaggedRow<TV> hw;
            if (t < nhalo) hw.load(ex, hp[0]);
            double v = 0.0;
#pragma unroll
            for (int q = 0; q < kPer; ++q) v += __builtin_bit_cast(double, u[q]);
            v = sum_mod8(v);
            if (lane < kResWords) wsum[wave * kResWords + lane] = v;
            __syncthreads();
            if (gave_up) return;
            const double s7 = sum_mod8(wsum[lane]);  // kWaves * kResWords == 64
            double sm[7];
#pragma unroll
            for (int j = 0; j < 7; ++j) sm[j] = read_lane(s7, j);
            const double alpha = sm[4] / sm[0];
            const double rr = sm[1] - 2.0 * alpha * sm[2] + alpha * alpha * sm[3];
            const double rz = sm[4] - 2.0 * alpha * sm[5] + alpha * alpha * sm[6];
            const bool conv = rr < threshold;
            const TV al = (TV)alpha;
            if (conv || k >= max_iter) {
                if (t < nrows) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) x_out[3 * (int64_t)node + c] = X.get(t, c) + al * own_p(t, c);
                    const TV none[3] = {0, 0, 0};
                    put_row(ring(0), row0 + t, none, 0u);
                    put_row(ring(1), row0 + t, none, 0u);
                }
                if ((int)blockIdx.x == wg.x && t == 0) {
                    sc->rr = rr;
                    sc->err = sqrt(fmax(rr, 0.0) / sc->bb);
                    sc->iters = conv ? k - 1 : k;
                    sc->converged = conv ? 1 : 0;
                    sc->done = 1;
                }
                return;
            }
            const TV be = (TV)(rz / sm[4]);
            if (t < nrows) {
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const TV p = own_p(t, c);
                    const TV z = Z.get(t, c) - al * Wv.get(t, c);
                    R.set(t, c, R.get(t, c) - al * Q.get(t, c));
                    X.set(t, c, X.get(t, c) + al * p);
                    Z.set(t, c, z);
                    po[c] = z + be * p;
                    P[3 * t + c] = po[c];
                }
            }
            // waits for a halo column's w of this iteration to be there
            auto arrive = [&](bool mine, int pos) {
                for (;;) {
                    const bool late = mine && !hw.is((unsigned)k);
                    if (!__any(late)) break;
                    if (too_long()) {
                        put(&sc->pad, 1);
                        gave_up = 1;
                        break;
                    }
                    asm volatile("" ::: "memory");  // loaded anew
                    if (late) hw.load(ex, pos);
                }
            };
            arrive(t < nhalo, hp[0]);
            if (t < nhalo) {
                const int j = 3 * (nrows + t);
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const TV z = ZH.get(t, c) - al * hw.get(c);
                    ZH.set(t, c, z);
                    ph[c] = z + be * (kRegs ? ph[c] : P[j + c]);
                    P[j + c] = ph[c];
                }
            }
            if (nhalo > kResThreads) {
                const bool mine = t + kResThreads < nhalo;
                if (mine) hw.load(ex, hp[1]);
                arrive(mine, hp[1]);
                if (mine) {
                    const int j = 3 * (nrows + kResThreads + t);
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const TV z = ZF.get(t, c) - al * hw.get(c);
                        ZF.set(t, c, z);
                        P[j + c] = z + be * P[j + c];
                    }
                }
            }
            __syncthreads();
            if (gave_up) return;
        }
        // q = S p: this lane's blocks, then the row's lanes in order
        {
            TV y0 = 0, y1 = 0, y2 = 0;
#pragma unroll
            for (int s = 0; s < (NB + 1) / 2; ++s) asm volatile("" : "+v"(cpk[s]));  // not unpacked ahead of the loop over k
            // the columns' p is read kAhead blocks ahead of its products: two waves per SIMD do not hide the LDS latency
            constexpr int kAhead = own_in_registers<TV, NB>() ? 3 : 2;
            TV pb[kAhead][3];
            auto fetch = [&](int s) {
                const TV* pc = (const TV*)((const char*)P + ((s & 1) ? cpk[s / 2] >> 16 : cpk[s / 2] & 0xffffu));
#pragma unroll
                for (int c = 0; c < 3; ++c) pb[s % kAhead][c] = pc[c];
            };
#pragma unroll
            for (int s = 0; s < kAhead; ++s) fetch(s);
#pragma unroll
            for (int s = 0; s < NB; ++s) {
                const TV p0 = pb[s % kAhead][0], p1 = pb[s % kAhead][1], p2 = pb[s % kAhead][2];
                if (s + kAhead < NB) fetch(s + kAhead);
                y0 = fma(m[s][0], p0, y0);
                y1 = fma(m[s][3], p0, y1);
                y2 = fma(m[s][6], p0, y2);
                y0 = fma(m[s][1], p1, y0);
                y1 = fma(m[s][4], p1, y1);
                y2 = fma(m[s][7], p1, y2);
                y0 = fma(m[s][2], p2, y0);
                y1 = fma(m[s][5], p2, y1);
                y2 = fma(m[s][8], p2, y2);
            }
            part[pi] = y0;
            part[pi + 1] = y1;
            part[pi + 2] = y2;
        }
        __syncthreads();
        double acc[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        {
            TV y[3] = {0, 0, 0}, w[3];
            for (int l = l01 & 0xffff; l < l01 >> 16; ++l)
#pragma unroll
                for (int c = 0; c < 3; ++c) y[c] += part[3 * l + c];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                if constexpr (kBlockPc) w[c] = (D.get(t, 3 * c) * y[0] + D.get(t, 3 * c + 1) * y[1]) + D.get(t, 3 * c + 2) * y[2];
                else w[c] = D.get(t, c) * y[c];
            }
            if (t < nrows) put_row(ring(k), row0 + t, w, (unsigned)k + 1u);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                Q.set(t, c, y[c]);
                Wv.set(t, c, w[c]);
                const double dr = (double)R.get(t, c), dy = (double)y[c], dz = (double)Z.get(t, c);
                acc[0] += (double)own_p(t, c) * dy;
                acc[1] += dr * dr;
                acc[2] += dr * dy;
                acc[3] += dy * dy;
                acc[4] += dr * dz;
                acc[5] += dy * dz;
                acc[6] += dy * (double)w[c];
            }
        }
        double s0, s1;
        wave_totals8(acc, s0, s1);
        if ((lane & 15) == 0) {
            rsum[wave * kResWords + (lane >> 3)] = s0;
            rsum[wave * kResWords + (lane >> 3) + 1] = s1;
        }
        __syncthreads();
        if (t < kResWords) {
            double s = 0.0;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) s += rsum[w * kResWords + t];
            put(&a.slots[((k & (kResRing - 1)) * kResMaxGroups + blockIdx.x) * kResWords + t], sum_word(s));
            put(&a.slots[(((k + 2) & (kResRing - 1)) * kResMaxGroups + blockIdx.x) * kResWords + t], kResEmpty);
        }
    }
}

// At most 512 own rows and 1,024 halo columns: their byte offsets fit 16 bits and everything fits 160 KB of LDS.
static_assert(lds_bytes<double, 10>() <= 158 * 1024 && lds_bytes<float, 20>() <= 158 * 1024, "LDS of a workgroup");
static_assert((kResMaxCols + 1) * 3 * sizeof(double) <= 65536, "column offsets");

template <typename TV, int NB>
void launch_nb(const ResidentArgs& a, hipStream_t s, int wgs) {
    constexpr size_t lds = lds_bytes<TV, NB>();
    static const hipError_t attr = hipFuncSetAttribute((const void*)cg_resident_kernel<TV, NB>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, 158 * 1024);
    if (attr != hipSuccess) throw std::runtime_error("cg_resident_kernel: LDS size refused");
    launch_k((cg_resident_kernel<TV, NB>), dim3(wgs), dim3(kResThreads), (uint32_t)lds, s, a);
}

// Blocks per lane, smallest first: the smallest that fits the CUs is taken, as short lane loops over many CUs beat long
// ones over few (whole steps, FP64 / FP32 + refinement: 21x18x20 cubes 181 us with 4 blocks against 213 with 7 and 222
// with 10 / 191 with 7, 198 with 10, 225 with 20; 30^3 260, 269, 285 / 256, 265, 290). The largest fill a lane's 256
// registers, 180 of them with blocks; in FP64 with 10 the compiler spills 8 others (20 bytes a lane).
constexpr int kNb64[] = {4, 7, 10};
constexpr int kNb32[] = {7, 10, 20};

// A start of several columns: blocks of dofs x columns.
__global__ __launch_bounds__(256) void columns_init_kernel(int n, const double* __restrict__ b,
                                                           const uint8_t* __restrict__ mask,
                                                           const int* __restrict__ diagblk, const double* __restrict__ S,
                                                           double* __restrict__ x, double* __restrict__ r,
                                                           double* __restrict__ z, double* __restrict__ dinv,
                                                           double* __restrict__ partial) {
    __shared__ double lds[8];
    const int col = blockIdx.y;
    double bb = 0.0, rz = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int I = i / 3, db = diagblk[I];
        const double s = db >= 0 ? S[9 * (int64_t)db + 4 * (i - 3 * I)] : 0.0;
        const double d = s != 0.0 ? 1.0 / s : 1.0;
        if (col == 0) dinv[i] = d;
        const int64_t o = (int64_t)col * n + i;
        const double bi = mask[i] ? 0.0 : b[o];
        const double zi = d * bi;
        x[o] = 0.0;
        r[o] = bi;
        z[o] = zi;
        bb += bi * bi;
        rz += bi * zi;
    }
    block_sum2(bb, rz, lds);
    if (threadIdx.x == 0) {
        partial[2 * kResColumnBlocks * col + blockIdx.x] = bb;
        partial[2 * kResColumnBlocks * col + kResColumnBlocks + blockIdx.x] = rz;
    }
}

// The columns' scalars (one wave each) and the published words emptied.
__global__ __launch_bounds__(64) void columns_setup_kernel(const double* __restrict__ partial, double tol,
                                                           CgScalars* __restrict__ sc,
                                                           unsigned long long* __restrict__ slots) {
    static_assert(kResColumnBlocks == 64, "one partial a lane");
    const int col = blockIdx.x;
    for (size_t i = col * 64 + threadIdx.x; i < kResSlotWords; i += gridDim.x * 64) slots[i] = kResEmpty;
    const double bb = wave_total(partial[2 * kResColumnBlocks * col + threadIdx.x]);
    const double rz = wave_total(partial[2 * kResColumnBlocks * col + kResColumnBlocks + threadIdx.x]);
    if (threadIdx.x != 0) return;
    CgScalars c = {};
    c.bb = bb;
    c.rz[0] = rz;
    c.threshold = fmax(tol * tol * bb, 2.2250738585072014e-308);
    c.rr = bb;
    if (bb == 0.0 || bb < c.threshold) {  // a zero column, or x = 0 already meets the test
        c.done = 1;
        c.converged = 1;
    }
    sc[col] = c;
}

}  // namespace

void launch_resident_columns(int num_nodes, int count, const double* b, const uint8_t* mask, const int* diagblk,
                             const double* S, double tol, double* x, double* r, double* z, double* dinv, double* partial,
                             CgScalars* sc, unsigned long long* slots, hipStream_t s) {
    launch_k(columns_init_kernel, dim3(kResColumnBlocks, count), dim3(256), 0, s, 3 * num_nodes, b, mask, diagblk, S, x, r,
             z, dinv, partial);
    launch_k(columns_setup_kernel, dim3(count), dim3(64), 0, s, (const double*)partial, tol, sc, slots);
}

void launch_cg_resident(const ResidentArgs& a, bool fp32, hipStream_t s, int wgs) {
    if (wgs == 0) wgs = a.t.groups * a.solves;
    if (wgs < 1 || wgs > kResMaxGroups) throw std::invalid_argument("one-launch CG: too many workgroups");
    if (fp32) {
        switch (a.t.nb) {
            case 7: return launch_nb<float, 7>(a, s, wgs);
            case 10: return launch_nb<float, 10>(a, s, wgs);
            case 20: return launch_nb<float, 20>(a, s, wgs);
        }
    } else {
        switch (a.t.nb) {
            case 4: return launch_nb<double, 4>(a, s, wgs);
            case 7: return launch_nb<double, 7>(a, s, wgs);
            case 10: return launch_nb<double, 10>(a, s, wgs);
        }
    }
    throw std::invalid_argument("no resident CG kernel for this plan");
}

namespace {

// Host threads for n nodes' worth of work (a mesh of a few thousand nodes is partitioned faster than a thread starts).
int host_threads(int64_t n) {
    return (int)std::max<int64_t>(1, std::min<int64_t>({8, (int64_t)std::thread::hardware_concurrency(), n / 4096}));
}

// work() on that many threads, this one among them.
template <typename Work>
void on_threads(int threads, const Work& work) {
    std::vector<std::future<void>> others;
    for (int i = 1; i < threads; ++i) others.push_back(std::async(std::launch::async, work));
    work();
    for (auto& o : others) o.get();
}

// Splits order[i0, i1) into `parts` compact sets by recursive bisection along the longest extent; ends[p] is the end of set
// p. Halves of large sets go to threads of their own.
void bisect(int32_t* order, const double* x0, int64_t i0, int64_t i1, int parts, int64_t* ends, int threads) {
    if (parts <= 1) {
        ends[0] = i1;
        return;
    }
    double lo[3], hi[3];
    for (int c = 0; c < 3; ++c) lo[c] = hi[c] = i0 < i1 ? x0[3 * (int64_t)order[i0] + c] : 0.0;
    for (int64_t i = i0; i < i1; ++i)
        for (int c = 0; c < 3; ++c) {
            const double v = x0[3 * (int64_t)order[i] + c];
            lo[c] = std::min(lo[c], v);
            hi[c] = std::max(hi[c], v);
        }
    int ax = 0;
    for (int c = 1; c < 3; ++c)
        if (hi[c] - lo[c] > hi[ax] - lo[ax]) ax = c;
    const int left = parts / 2;
    const int64_t mid = i0 + (i1 - i0) * left / parts;
    std::nth_element(order + i0, order + mid, order + i1, [&](int32_t p, int32_t q) {
        const double a = x0[3 * (int64_t)p + ax], b = x0[3 * (int64_t)q + ax];
        return a < b || (a == b && p < q);
    });
    auto first = [=] { bisect(order, x0, i0, mid, left, ends, threads / 2); };
    std::future<void> half;
    if (threads > 1) half = std::async(std::launch::async, first);
    else first();
    bisect(order, x0, mid, i1, parts - left, ends + left, threads - threads / 2);
    if (half.valid()) half.get();
}

// One workgroup's rows order[i0, i1): its lanes and halo into the plan. False when it does not fit. local: -1 per node, and
// left so, from node n0 on.
bool plan_group(ResidentPlan& plan, int g, int64_t i0, int64_t i1, int64_t n0, const int32_t* rp, const int32_t* ci,
                std::vector<int32_t>& local_of, std::vector<int32_t>& halo) {
    struct Share {  // a lane's blocks of one row
        int deg, chunk, cnt, part;
        int32_t k0;
    };
    const int nb = plan.nb, nrows = (int)(i1 - i0);
    int32_t* local = local_of.data() - n0;
    const int32_t* order = plan.row_node.data();
    if (nrows > kResThreads) return false;
    std::vector<Share> shares;
    for (int64_t i = i0; i < i1; ++i) local[order[i]] = (int32_t)(i - i0);
    for (int64_t i = i0; i < i1; ++i) {
        plan.row_lane[(size_t)g * (kResThreads + 1) + (i - i0)] = (uint16_t)std::min<size_t>(shares.size(), kResThreads);
        const int32_t I = order[i], deg = rp[I + 1] - rp[I], lanes = std::max(1, (deg + nb - 1) / nb);
        int32_t k = rp[I];
        for (int q = 0; q < lanes; ++q) {  // differing by at most one block
            const int cnt = deg / lanes + (q < deg % lanes ? 1 : 0);
            shares.push_back({deg, q, cnt, (int)shares.size(), k});
            k += cnt;
        }
        for (int32_t j = rp[I]; j < rp[I + 1]; ++j) {
            const int32_t J = ci[j];
            if (local[J] < 0) {
                local[J] = nrows + (int32_t)halo.size();
                halo.push_back(J);
            }
        }
    }
    const int parts = (int)shares.size();
    const bool fits = parts <= kResThreads && halo.size() <= 2 * (size_t)kResThreads;
    if (fits) {
        for (int r = nrows; r <= kResThreads; ++r) plan.row_lane[(size_t)g * (kResThreads + 1) + r] = (uint16_t)parts;
        // Neighbouring lanes take the same share of rows alike (as on a structured mesh), whose columns then lie at one
        // stride in LDS.
        std::stable_sort(shares.begin(), shares.end(), [](const Share& a, const Share& b) {
            return a.deg != b.deg ? a.deg < b.deg : a.chunk < b.chunk;
        });
        for (int lane = 0; lane < kResThreads; ++lane) {
            const size_t li = (size_t)g * kResThreads + lane;
            if (lane >= parts) {
                plan.lane_info[li] = (int32_t)lane << 8;  // no blocks; a part that no row reads
                continue;
            }
            const Share& sh = shares[lane];
            // a row without blocks (a node in no element) starts at 0: the kernel loads a first block all the same, and its
            // own place is past the operator's end where no later row has blocks
            plan.lane_k0[li] = sh.cnt > 0 ? sh.k0 : 0;
            plan.lane_info[li] = sh.cnt | sh.part << 8;
            for (int s = 0; s < sh.cnt; ++s)
                plan.cols[((size_t)g * nb + s) * kResThreads + lane] = (uint16_t)local[ci[sh.k0 + s]];
        }
    }
    for (int64_t i = i0; i < i1; ++i) local[order[i]] = -1;
    for (int32_t J : halo) local[J] = -1;
    return fits;
}

// The plan of nodes [n0, n0 + N) for nb blocks per lane and the given number of workgroups, made by `threads` host threads; empty
// when a workgroup would overflow.
ResidentPlan try_plan(int64_t n0, int64_t N, const int32_t* rp, const int32_t* ci, const double* x0, bool fp32, int nb,
                      int groups, int threads) {
    ResidentPlan plan;
    std::vector<int64_t> ends(groups + 1, 0);  // set g: [ends[g], ends[g + 1])
    plan.row_node.resize(N);
    std::iota(plan.row_node.begin(), plan.row_node.end(), (int32_t)n0);
    bisect(plan.row_node.data(), x0, 0, N, groups, ends.data() + 1, threads);
    plan.nb = nb;
    plan.lane_k0.assign((size_t)groups * kResThreads, 0);
    plan.lane_info.assign((size_t)groups * kResThreads, 0);
    plan.row_lane.assign((size_t)groups * (kResThreads + 1), 0);
    plan.cols.assign((size_t)groups * nb * kResThreads, kResMaxCols);
    std::vector<std::vector<int32_t>> halo(groups);
    std::atomic<int> next{0};
    std::atomic<bool> fits{true};
    auto work = [&] {
        std::vector<int32_t> local(N, -1);
        for (int g; fits && (g = next++) < groups;) {
            std::sort(plan.row_node.begin() + ends[g], plan.row_node.begin() + ends[g + 1]);
            if (!plan_group(plan, g, ends[g], ends[g + 1], n0, rp, ci, local, halo[g])) fits = false;
        }
    };
    on_threads(threads, work);
    if (!fits) return {};
    std::vector<int32_t> pos(N);  // rows of the partition, counted from n0 as the nodes are
    for (int64_t i = 0; i < N; ++i) pos[plan.row_node[i] - n0] = (int32_t)(n0 + i);
    for (int g = 0; g < groups; ++g) {
        plan.group.push_back(make_int4((int)(n0 + ends[g]), (int)(ends[g + 1] - ends[g]), (int)plan.halo_node.size(),
                                       (int)halo[g].size()));
        for (int32_t J : halo[g]) {
            plan.halo_node.push_back(J);
            plan.halo_pos.push_back(pos[J - n0]);
        }
    }
    const int bytes = 3 * (fp32 ? 4 : 8);
    for (auto& c : plan.cols) c = (uint16_t)(c * bytes);
    plan.groups = groups;
    return plan;
}

int64_t lanes_of(int64_t n0, int64_t n1, const int32_t* rp, int nb) {
    int64_t lanes = 0;
    for (int64_t I = n0; I < n1; ++I) lanes += std::max(1, (rp[I + 1] - rp[I] + nb - 1) / nb);
    return lanes;
}

constexpr int kResFill = kResThreads * 9 / 10;  // lanes asked of a workgroup: the sets' lanes differ by a few percent

// The plan of nodes [n0, n1) with nb blocks per lane on as few workgroups as take it, at most `most`.
ResidentPlan fit_plan(int64_t n0, int64_t n1, const int32_t* rp, const int32_t* ci, const double* x0, bool fp32, int nb,
                      int most, int threads) {
    const int64_t lanes = lanes_of(n0, n1, rp, nb);
    if (lanes > (int64_t)most * kResThreads) return {};
    for (int64_t groups = (lanes + kResFill - 1) / kResFill;; groups += std::max<int64_t>(1, groups / 16)) {
        ResidentPlan p = try_plan(n0, n1 - n0, rp, ci, x0, fp32, nb, (int)std::min<int64_t>(groups, most), threads);
        if (p.groups || groups >= most) return p;
    }
}

}  // namespace

ResidentPlan plan_resident(int64_t N, const int32_t* rp, const int32_t* ci, const double* x0, bool fp32, int num_cus) {
    const int most = std::min(num_cus, kResMaxGroups);
    if (N <= 0 || N > (int64_t)most * kResThreads) return {};
    for (int nb : fp32 ? kNb32 : kNb64) {
        ResidentPlan p = fit_plan(0, N, rp, ci, x0, fp32, nb, most, host_threads(N));
        if (p.groups) return p;
    }
    return {};
}

ResidentPlan plan_resident_batch(const std::vector<int64_t>& off, const int32_t* rp, const int32_t* ci, const double* x0,
                                 bool fp32, int num_cus) {
    const int most = std::min(num_cus, kResMaxGroups), M = (int)off.size() - 1;
    if (off[M] > kResMaxRows) return {};
    // Fewest launches, each weighed by the time of an iteration with that many blocks per lane (3.8, 5.0, 6.2 us measured
    // in FP64, 3.8, 4.2, 5.2 us in FP32): the launches of a batch run one after another.
    const double weight[2][3] = {{3.8, 5.0, 6.2}, {3.8, 4.2, 5.2}};
    int nb = 0;
    double least = 0.0;
    for (int i = 0; i < 3; ++i) {
        const int b = fp32 ? kNb32[i] : kNb64[i];
        int64_t groups = 0, left = 0;
        for (int m = 0; m < M; ++m) {
            const int64_t g = (lanes_of(off[m], off[m + 1], rp, b) + kResFill - 1) / kResFill;
            if (g <= most) groups += g;
            else left += g;  // solved with a launch per iteration
        }
        const double cost = weight[fp32][i] * (double)((groups + most - 1) / most) + 10.0 * (double)left;
        if (nb == 0 || cost < least) {
            nb = b;
            least = cost;
        }
    }
    ResidentPlan all;
    all.nb = nb;
    all.instances.assign(M, 0);
    std::vector<std::array<int, 3>> inst;  // groups, first group, instance
    all.row_node.resize(off[M]);
    std::iota(all.row_node.begin(), all.row_node.end(), 0);
    // an instance a thread, or a few large ones one after another by all threads (64 bodies of 25^3: 116 ms one after another by
    // one thread)
    const int threads = host_threads(off[M]);
    std::vector<ResidentPlan> plans(M);
    std::atomic<int> next{0};
    on_threads(M < threads ? 1 : threads, [&] {
        for (int m; (m = next++) < M;)
            plans[m] = fit_plan(off[m], off[m + 1], rp, ci, x0, fp32, nb, most, M < threads ? threads : 1);
    });
    for (int m = 0; m < M; ++m) {
        const ResidentPlan p = std::move(plans[m]);
        if (!p.groups) continue;
        all.instances[m] = 1;
        inst.push_back({p.groups, (int)all.group.size(), m});
        std::copy(p.row_node.begin(), p.row_node.end(), all.row_node.begin() + off[m]);
        for (int4 g : p.group) {
            g.z += (int)all.halo_node.size();
            all.group.push_back(g);
        }
        auto append = [](auto& to, const auto& from) { to.insert(to.end(), from.begin(), from.end()); };
        append(all.halo_node, p.halo_node);
        append(all.halo_pos, p.halo_pos);
        append(all.lane_k0, p.lane_k0);
        append(all.lane_info, p.lane_info);
        append(all.row_lane, p.row_lane);
        append(all.cols, p.cols);
    }
    all.groups = (int)all.group.size();
    // instances to launches, largest first into the first launch with room
    std::stable_sort(inst.begin(), inst.end(), [](const auto& a, const auto& b) { return a[0] > b[0]; });
    std::vector<std::vector<std::array<int, 3>>> launch;
    for (const auto& i : inst) {
        size_t l = 0;
        while (l < launch.size() && all.launches[l] + i[0] > most) ++l;
        if (l == launch.size()) {
            launch.emplace_back();
            all.launches.push_back(0);
        }
        launch[l].push_back(i);
        all.launches[l] += i[0];
    }
    for (const auto& l : launch) {
        int first = 0;
        for (const auto& i : l) {
            for (int g = 0; g < i[0]; ++g) all.wg.push_back(make_int4(first, i[0], i[1] + g, i[2]));
            first += i[0];
        }
    }
    return all;
}

}  // namespace femgpu
