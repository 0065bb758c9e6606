// The planner of columns_kernel and column_rows_kernel compiled on its own with a host compiler: for every shape given on
// the command line as "kind n_samples l_max bytes" quadruples one line of numbers, for an MI355X (160 KB of LDS per
// workgroup, 256 CUs): whether there is a plan, lanes per point, workgroups, threads, bytes of LDS, tiles, pad, the two
// offsets, for the vector-Jacobian product whether it is taken, and whether the kernel has l_max for a constant.
#include <cstdio>
#include <cstdlib>

#include "../sphericart_amd/csrc/sphx_columns.hpp"
#include "../sphericart_amd/csrc/sphx_plan.hpp"

int main(int argc, char** argv) {
    for (int i = 1; i + 3 < argc; i += 4) {
        const auto kind = static_cast<sphx::ColumnsKind>(std::atoi(argv[i]));
        const size_t n = static_cast<size_t>(std::atoll(argv[i + 1]));
        const int l_max = std::atoi(argv[i + 2]);
        const size_t elem = static_cast<size_t>(std::atoi(argv[i + 3]));
        (void)sphx::refresh_switches();
        sphx::ColumnsLaunch c{}, taken{};
        const bool there = sphx::plan_columns(kind, n, l_max, elem, 160 * 1024, 256, &c);
        sphx::VjpPlan other;
        bool by_columns = false;
        if (kind == sphx::COLUMNS_VJP && sphx::make_vjp_plan(n, l_max, elem, 160 * 1024, 256, &other) == 0) {
            by_columns = sphx::vjp_by_columns(n, l_max, elem, 160 * 1024, 256, other, &taken);
        }
        std::printf("%d %d %u %u %u %u %u %u %u %d %d\n", there, c.groups, c.workgroups, c.threads, c.lds_bytes, c.g.n_tiles,
                    c.g.pad, c.g.off_rows, c.g.off_sums, by_columns, there && c.fixed);
    }
    return 0;
}
