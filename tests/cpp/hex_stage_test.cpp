// Checks of the hexahedra's staging map without a GPU: where a node finds its elements' staged values.
#include "fem_hex.hpp"

#include <cstdio>

using namespace femgpu;

namespace {

int failures = 0;
void check(bool ok, const char* what) {
    std::printf("%s: %s\n", ok ? "ok" : "FAILED", what);
    failures += !ok;
}

uint64_t staged(uint64_t position, int corner) { return position / 64 * 24 * 64 + (uint64_t)(3 * corner) * 64 + position % 64; }

// The map holds, node by node, the corners of the positions' elements in the positions' order.
bool holds(const HexStageMap& m, int64_t nodes, const std::vector<int32_t>& conn, const std::vector<int>& order) {
    std::vector<std::vector<uint64_t>> want(nodes);
    for (size_t t = 0; t < order.size(); ++t)
        if (order[t] >= 0)
            for (int a = 0; a < 8; ++a) want[conn[8 * (size_t)order[t] + a]].push_back(staged(t, a));
    for (int64_t i = 0; i < nodes; ++i) {
        std::vector<uint64_t> got;
        for (int k = 0; k < m.slots; ++k)
            if (m.src[(size_t)k * nodes + i] != kNotStaged) got.push_back(m.src[(size_t)k * nodes + i]);
        if (!m.more_ptr.empty())
            for (int64_t j = m.more_ptr[i]; j < m.more_ptr[i + 1]; ++j) got.push_back(m.more[j]);
        if (got != want[i]) return false;
    }
    return true;
}

}  // namespace

int main() {
    {  // elements that share a node each: 1, 8, 9 and 1,000 elements at it
        for (int count : {1, 8, 9, 1000}) {
            const int64_t nodes = 1 + 7 * (int64_t)count;
            std::vector<int32_t> conn;
            std::vector<int> order;
            for (int e = 0; e < count; ++e) {
                for (int a = 0; a < 8; ++a) conn.push_back(a == e % 8 ? 0 : 1 + 7 * e + (a > e % 8 ? a - 1 : a));
                order.push_back(e);
                order.resize(order.size() + (e % 3 == 0 ? 63 : 0), -1);  // padding inside
            }
            const HexStageMap m = hex_stage_map(nodes, conn.data(), order);
            check(holds(m, nodes, conn, order), "every node's elements");
            check((int64_t)m.src.size() <= kStageSlots * nodes && (int64_t)m.more.size() == std::max(0, count - kStageSlots),
                  "a node of many elements adds its own only");
        }
    }
    {  // 90 million and 2^27 positions: more than 2^31 staged values
        const std::vector<int32_t> conn{0, 1, 2, 3, 4, 5, 6, 7};
        for (size_t positions : {(size_t)90000000, (size_t)1 << 27}) {
            std::vector<int> order(positions, -1);
            order.back() = 0;
            const HexStageMap m = hex_stage_map(8, conn.data(), order);
            check(holds(m, 8, conn, order), "the last position of a large mesh");
        }
    }
    std::printf("%d failed\n", failures);
    return failures != 0;
}
