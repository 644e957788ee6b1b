// Checks csrc/items.h on the host: every workgroup order is a permutation, every element of a
// set of tensors is in exactly one work item at every chunk size, and a bound on the update's
// grid allows the same lanes whatever an instance's workgroups are.
// Prints "items_check: ok" when nothing differs.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "items.h"

static int failures = 0;

#define CHECK(cond, ...)              \
    do {                              \
        if (!(cond)) {                \
            ++failures;               \
            std::printf(__VA_ARGS__); \
            std::printf("\n");        \
        }                             \
    } while (0)

template <int kRun>
static void check_order() {
    const int64_t group = 8 * kRun;
    for (int64_t n : {int64_t(1), group - 1, group, group + 1, 3 * group, 9 * group + 5}) {
        std::vector<char> seen(n, 0);
        for (int64_t w = 0; w < n; ++w) {
            const int64_t it = item_order<kRun>(w, n);
            CHECK(it >= 0 && it < n && !seen[it], "run %d, n %lld: item %lld", kRun, (long long)n,
                  (long long)it);
            if (it >= 0 && it < n) seen[it] = 1;
        }
    }
}

// Tables as the kernels read them, with host memory in place of device memory.
struct HostTable {
    std::vector<int64_t> numel;
    std::vector<mi_adamw_chunk> chunks;
    HostTable(std::vector<int64_t> sizes, int64_t chunk_elems) : numel(sizes) {
        for (size_t r = 0; r < sizes.size(); ++r)
            for (int64_t k = 0; k * chunk_elems < sizes[r]; ++k)
                chunks.push_back({static_cast<int32_t>(r), static_cast<int32_t>(k)});
    }
    void get(int64_t c, int64_t chunk_elems, mi_adamw_tensor&, int64_t& begin, int64_t& end,
             int32_t& row) const {
        row = chunks[c].tensor;
        begin = chunks[c].index * chunk_elems;
        end = begin + chunk_elems < numel[row] ? begin + chunk_elems : numel[row];
    }
};

template <int kTile>
static void check_cover() {
    for (int64_t chunk : {4096, 12288, 65536}) {
        const HostTable table({1, 3, 768, kTile - 1, kTile, kTile + 1, 4095, 4097, chunk,
                               chunk + 1, 3 * chunk + 5 * kTile + 2},
                              chunk);
        const Items items = items_of(table.chunks.size(), chunk, kTile);
        std::vector<std::vector<char>> seen;
        for (int64_t n : table.numel) seen.emplace_back(n, 0);
        for (int64_t it = 0; it < items.n; ++it) {
            mi_adamw_tensor t{};
            int64_t begin = 0, end = 0;
            int32_t row = 0;
            if (!items.get<kTile>(table, it, t, begin, end, row)) continue;
            CHECK(begin < end && end - begin <= kTile && begin % 4 == 0, "tile %d, chunk %lld",
                  kTile, (long long)chunk);
            for (int64_t i = begin; i < end; ++i) ++seen[row][i];
        }
        for (size_t r = 0; r < seen.size(); ++r)
            for (char s : seen[r])
                if (s != 1) {
                    CHECK(false, "tile %d, chunk %lld, tensor %zu", kTile, (long long)chunk, r);
                    break;
                }
    }
}

static void check_bound() {
    const int64_t many = int64_t(1) << 22;
    for (int threads : {256, 512, 1024}) {
        for (int32_t bound : {1, 7, 512, 1025}) {
            CHECK(int64_t(update_grid(many, bound, threads)) * threads == int64_t(bound) * 1024,
                  "bound %d, %d lanes: %u workgroups", bound, threads,
                  update_grid(many, bound, threads));
            CHECK(update_grid(1, bound, threads) == 1, "one item");
        }
        CHECK(update_grid(5000, 0, threads) == 5000, "no bound");
        CHECK(update_grid(5000, 0x7fffffff, threads) == 5000, "the largest bound");
        CHECK(int64_t(update_grid(int64_t(1) << 40, 0, threads)) * threads <= 0x7fffffff,
              "the largest launch");
    }
}

int main() {
    check_order<16>();
    check_order<32>();
    check_order<128>();
    check_cover<1024>();
    check_cover<2048>();
    check_cover<4096>();
    check_bound();
    if (failures) return 1;
    std::printf("items_check: ok\n");
    return 0;
}
