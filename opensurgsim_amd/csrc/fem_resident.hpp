// Conjugate gradients with the operator held on the chip: one launch runs a whole solve (see fem_resident.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "fem_kernels.hpp"

namespace femgpu {

constexpr int kResThreads = 512;      // lanes of a workgroup, each holding up to nb blocks of one block row
constexpr int kResMaxGroups = 256;    // workgroups of a solve (one per CU)
constexpr int kResWords = 8;          // published words per workgroup and iteration (7 sums, 1 spare)
constexpr int kResRing = 4;           // iterations whose published sums are kept apart
constexpr int kResRowBytes64 = 48, kResRowBytes32 = 24;  // a node's w in the exchange, FP64 and FP32
constexpr int64_t kResMaxRows = INT32_MAX / kResRowBytes64;  // nodes of a batch: the exchange is addressed by 32-bit offsets
constexpr size_t kResSlotWords = (size_t)kResRing * kResMaxGroups * kResWords;

// Partition of the block rows over the workgroups of a solve, with every lane's blocks and local columns.
struct ResidentTables {
    int groups = 0;      // workgroups (of one solve; of all instances of a batch)
    int nb = 0;          // blocks per lane
    int rows = 0;        // rows of the partition
    // all pointers into one device allocation
    const int4* group = nullptr;        // first row (partition order), rows, first halo entry, halo columns
    const int4* wg = nullptr;           // batch: first workgroup and workgroups of its solve in the launch, group, instance
    const int* row_node = nullptr;      // node of each row, partition order
    const int* halo_node = nullptr;     // node of each halo column
    const int* halo_pos = nullptr;      // and its row in partition order
    const int* lane_k0 = nullptr;       // first block of each lane
    const int* lane_info = nullptr;     // its blocks (0 .. nb, 8 bits) and where its part of the row goes
    const uint16_t* row_lane = nullptr; // first part of each row, kResThreads + 1 per workgroup
    const uint16_t* cols = nullptr;     // [group][nb][lane] byte offsets of the local columns (own rows, then halo)
};

// Host side of the partition: empty (groups == 0) when the system does not fit the device's CUs.
struct ResidentPlan {
    int groups = 0, nb = 0;
    std::vector<int4> group, wg;
    std::vector<int32_t> row_node, halo_node, halo_pos, lane_k0, lane_info;
    std::vector<uint16_t> row_lane, cols;
    std::vector<int> launches;        // batch: workgroups of each launch (wg holds them one launch after another)
    std::vector<uint8_t> instances;   // batch: 1 for the instances the plan solves
};
ResidentPlan plan_resident(int64_t num_nodes, const int32_t* rowptr, const int32_t* colidx, const double* x0, bool fp32,
                           int num_cus);
// Independent instances (nodes [offsets[i], offsets[i + 1])), as many to a launch as fit the CUs together.
ResidentPlan plan_resident_batch(const std::vector<int64_t>& offsets, const int32_t* rowptr, const int32_t* colidx,
                                 const double* x0, bool fp32, int num_cus);

struct ResidentArgs {
    ResidentTables t;
    const void* S;           // 9 TV per block
    const void* r;           // r_0, z_0 and x_0 by DOF
    const void* z;
    void* x;                 // solution by DOF
    const void* dinv;        // FP64: diagonal preconditioner (one value per DOF); FP32: 3x3 blocks (9 per node)
    void* exch;              // [2][nodes] w by iteration parity, partition order, kResRowBytes64 / 32 a node; zero at the first launch
    unsigned long long* slots;  // kResSlotWords words, all kResEmpty at launch
    CgScalars* sc;
    int max_iter;            // at least 1
    const int* max_iters = nullptr;  // batch: per instance instead
    int solves = 1;          // solves of one operator in the launch: r, z, x of solve i at i * stride values, sc + i
    int64_t stride = 0;
    long long wait_ticks;    // the longest wait for another workgroup, in ticks of the 100 MHz clock
};
constexpr unsigned long long kResEmpty = ~0ull;  // a word not published yet

// Workgroups of the launch: t.groups for each of `solves`; `wgs` for a launch of a batch (t.wg).
void launch_cg_resident(const ResidentArgs& a, bool fp32, hipStream_t s, int wgs = 0);

// The start of `count` FP64 solves of columns of b (n values each): x = 0, r = b with boundary rows zero, z = r / diag(S)
// (1 where the diagonal is 0), the scalars at tolerance tol, the published words emptied.
// partial: 2 * kResColumnBlocks doubles a column.
constexpr int kResColumnBlocks = 64;
constexpr int kResMaxColumns = 64;  // columns of one launch
void launch_resident_columns(int num_nodes, int count, const double* b, const uint8_t* mask, const int* diagblk,
                             const double* S, double tol, double* x, double* r, double* z, double* dinv, double* partial,
                             CgScalars* sc, unsigned long long* slots, hipStream_t s);

}  // namespace femgpu
