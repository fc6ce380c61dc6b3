// Checks of the one-launch CG's host side, without a GPU: the partition of an operator over workgroups.
#include "fem_resident.hpp"

#include <algorithm>
#include <cstdio>
#include <numeric>

using namespace femgpu;

namespace {

int failures = 0;
#define CHECK(cond, ...)                                     \
    do {                                                     \
        if (!(cond)) {                                       \
            if (++failures <= 20) {                          \
                std::printf("FAILED %s: ", #cond);           \
                std::printf(__VA_ARGS__);                    \
                std::printf("\n");                           \
            }                                                \
        }                                                    \
    } while (0)

// Block rows of a grid of nodes joined to their neighbours (up to 27 blocks a row), unused nodes (empty rows) put where
// asked: before, in the middle of, and after the used ones.
struct Mesh {
    std::vector<int32_t> rp{0}, ci;
    std::vector<double> x0;
    int64_t nodes() const { return (int64_t)rp.size() - 1; }
    void unused(int count) {
        for (int i = 0; i < count; ++i) {
            rp.push_back((int32_t)ci.size());
            x0.insert(x0.end(), {0.5 * i, -1.0, 2.0});
        }
    }
    void grid(int nx, int ny, int nz, int unused_inside) {
        const int split = nx * ny * nz / 2;  // the unused nodes' place among the grid's
        const int32_t base = (int32_t)nodes();
        auto id = [&](int i, int j, int k) {
            const int n = (i * ny + j) * nz + k;
            return base + n + (n >= split ? unused_inside : 0);
        };
        for (int i = 0; i < nx; ++i)
            for (int j = 0; j < ny; ++j)
                for (int k = 0; k < nz; ++k) {
                    if ((i * ny + j) * nz + k == split) unused(unused_inside);
                    for (int a = std::max(0, i - 1); a <= std::min(nx - 1, i + 1); ++a)
                        for (int b = std::max(0, j - 1); b <= std::min(ny - 1, j + 1); ++b)
                            for (int c = std::max(0, k - 1); c <= std::min(nz - 1, k + 1); ++c) ci.push_back(id(a, b, c));
                    rp.push_back((int32_t)ci.size());
                    x0.insert(x0.end(), {1.0 * i, 1.0 * j, 1.0 * k});
                }
    }
};

// The plan covers the rows [n0, n1) of every planned instance, each row's blocks once and in order, and no lane reads a
// block that is not there: a lane without blocks still loads its first one.
void check_plan(const char* name, const Mesh& m, const ResidentPlan& p, int64_t covered) {
    const int64_t blocks = m.rp.back();
    CHECK(p.groups == (int)p.group.size(), "%s", name);
    CHECK((int64_t)p.lane_k0.size() == (int64_t)p.groups * kResThreads, "%s", name);
    for (size_t li = 0; li < p.lane_k0.size(); ++li) {
        const int64_t cnt = p.lane_info[li] & 0xff;
        CHECK(p.lane_k0[li] >= 0 && p.lane_k0[li] + std::max<int64_t>(cnt, 1) <= blocks, "%s: lane %zu reads block %d of %lld",
              name, li, p.lane_k0[li], (long long)blocks);
    }
    std::vector<int32_t> seen(m.nodes(), 0);
    int64_t rows = 0;
    for (int g = 0; g < p.groups; ++g) {
        const int4 info = p.group[g];
        std::vector<int64_t> lane_of_part(kResThreads, -1);
        for (int lane = 0; lane < kResThreads; ++lane)
            lane_of_part[p.lane_info[(size_t)g * kResThreads + lane] >> 8] = (int64_t)g * kResThreads + lane;
        for (int r = 0; r < info.y; ++r, ++rows) {
            const int32_t node = p.row_node[info.x + r];
            ++seen[node];
            const uint16_t* rl = &p.row_lane[(size_t)g * (kResThreads + 1) + r];
            int64_t k = m.rp[node];
            for (int part = rl[0]; part < rl[1]; ++part) {
                const int64_t li = lane_of_part[part], cnt = li < 0 ? 0 : p.lane_info[li] & 0xff;
                CHECK(li >= 0 && (cnt == 0 || p.lane_k0[li] == k), "%s: node %d", name, node);
                k += cnt;
            }
            CHECK(k == m.rp[node + 1], "%s: node %d", name, node);
        }
    }
    CHECK(rows == covered, "%s: %lld rows", name, (long long)rows);
    for (int32_t s : seen) CHECK(s <= 1, "%s", name);
}

void unused_nodes() {
    for (int where = 0; where < 3; ++where)
        for (int count : {1, 5})
            for (bool fp32 : {false, true}) {
                Mesh m;
                if (where == 0) m.unused(count);
                m.grid(6, 5, 7, where == 1 ? count : 0);
                if (where == 2) m.unused(count);
                const ResidentPlan p = plan_resident(m.nodes(), m.rp.data(), m.ci.data(), m.x0.data(), fp32, 256);
                CHECK(p.groups > 0, "place %d", where);
                check_plan("one", m, p, m.nodes());

                Mesh b;  // the same three times, and an instance of unused nodes alone
                std::vector<int64_t> off{0};
                for (int i = 0; i < 3; ++i) {
                    if (where == 0) b.unused(count);
                    b.grid(3 + i, 5, 7 - i, where == 1 ? count : 0);
                    if (where == 2) b.unused(count);
                    off.push_back(b.nodes());
                }
                b.unused(2);
                off.push_back(b.nodes());
                const ResidentPlan q = plan_resident_batch(off, b.rp.data(), b.ci.data(), b.x0.data(), fp32, 256);
                CHECK(q.groups > 0, "place %d", where);
                check_plan("batch", b, q, b.nodes());
            }
}

// Batches planned by several host threads: an instance a thread (24 of them), and all threads on each of a few.
void batches_on_threads() {
    for (int count : {24, 3})
        for (bool fp32 : {false, true}) {
            Mesh m;
            std::vector<int64_t> off{0};
            for (int i = 0; i < count; ++i) {
                if (count == 3) m.grid(20, 19 + i, 21, 0);
                else m.grid(9 + i % 5, 12, 11 + i % 3, 0);
                off.push_back(m.nodes());
            }
            const ResidentPlan p = plan_resident_batch(off, m.rp.data(), m.ci.data(), m.x0.data(), fp32, 256);
            check_plan("threads", m, p, m.nodes());
            CHECK((int)p.wg.size() == p.groups && std::accumulate(p.launches.begin(), p.launches.end(), 0) == p.groups, "%d", count);
            for (uint8_t planned : p.instances) CHECK(planned, "%d", count);
        }
}

// A batch of more nodes than the exchange addresses: one instance that would fit the chip beside unused nodes.
void batch_beyond_the_exchange() {
    for (int64_t nodes : {kResMaxRows, kResMaxRows + 1}) {
        Mesh m;
        m.grid(3, 3, 3, 0);
        const std::vector<int64_t> off{0, m.nodes(), nodes};
        m.rp.resize(nodes + 1, m.rp.back());
        const ResidentPlan p = plan_resident_batch(off, m.rp.data(), m.ci.data(), m.x0.data(), false, 256);
        CHECK((p.groups > 0) == (nodes == kResMaxRows), "%lld nodes", (long long)nodes);
    }
}

}  // namespace

int main() {
    unused_nodes();
    batches_on_threads();
    batch_beyond_the_exchange();
    std::printf("%s: %d failed checks\n", failures ? "FAILED" : "ok", failures);
    return failures != 0;
}
