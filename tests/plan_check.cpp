// CPU check of the products' plan and placement in weed_amd/csrc/matmul_plan.h (built and run by tests/test_matmul_plan_cpu.py with
// g++; no GPU involved).  Without arguments: every tile, k range and product goes to exactly one workgroup.  With arguments M N K batch
// most off_grid b_along_k, seven numbers a product: what it is planned as, one line each.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../weed_amd/csrc/matmul_plan.h"

using namespace weedmm;

static bool places_all(uint32_t m_tiles, uint32_t n_tiles, uint32_t zs)
{
    const uint32_t wgs = m_tiles * n_tiles * zs;
    std::vector<char> seen(wgs, 0);
    for (uint32_t wg = 0; wg < wgs; ++wg) {
        uint32_t mt, nt, z;
        split_place(wg, wgs, m_tiles, n_tiles, mt, nt, z);
        if (mt >= m_tiles || nt >= n_tiles || z >= zs) {
            return false;
        }
        char &s = seen[(z * n_tiles + nt) * m_tiles + mt];
        if (s) {
            return false;
        }
        s = 1;
    }
    return true;
}

int main(int argc, char **argv)
{
    if (argc == 1) {
        for (uint32_t m_tiles = 1; m_tiles <= 40; ++m_tiles) {
            for (uint32_t n_tiles = 1; n_tiles <= 40; n_tiles += 1 + n_tiles / 9) {
                for (uint32_t zs : { 1U, 2U, 3U, 7U, 64U }) {
                    if (!places_all(m_tiles, n_tiles, zs)) {
                        std::printf("FAILED at %u x %u tiles, %u\n", m_tiles, n_tiles, zs);
                        return 1;
                    }
                }
            }
        }
        std::printf("OK\n");
        return 0;
    }
    for (int i = 1; i + 6 < argc; i += 7) {
        const auto arg = [&](int x) { return (uint32_t)std::strtoul(argv[i + x], nullptr, 10); };
        const uint32_t M = arg(0), N = arg(1), K = arg(2), batch = arg(3), most = arg(4);
        const bool off_grid = arg(5), b_along_k = arg(6);
        TilePlan plan{ kTile, 1, 0, 0.0 };
        bool strips = false;
        if ((uint64_t)M * N * K * batch >= (1ull << 30)) {
            plan = plan_tiles(M, N, K, batch, most, off_grid);
            strips = has_strips(M, N, K, batch) && strips_beat(plan, M, N, K, b_along_k, most, off_grid);
        } else if (batch == 1 && K >= 256) {
            const uint32_t s = std::min(most, choose_k_splits((uint64_t)tiles_of(M, kTile) * tiles_of(N, kTile), K));
            plan.k_per_split = s > 1 ? ((K + s - 1) / s + kSlice - 1) / kSlice * kSlice : 0U;
            plan.splits = s > 1 ? tiles_of(K, plan.k_per_split) : 1U;
        }
        const uint32_t wgs = tiles_of(M, plan.tile) * tiles_of(N, plan.tile) * (plan.splits > 1 ? plan.splits : batch);
        std::printf("tile %u splits %u wgs %u placed %d three %d strips %d\n", plan.tile, plan.splits, wgs, wgs >= kPlaced,
                    plan.tile == kTile && three_per_unit(K, plan.k_per_split, wgs), strips);
    }
    return 0;
}
