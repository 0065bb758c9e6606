// The tables of sphx_plan_shapes.hpp against the planner, on an MI355X (160 KB of LDS per workgroup, 256 CUs): prints every
// row, with one of its l_max, that no call without overrides is planned by, whatever its number of points.
#include <cmath>
#include <cstdio>
#include <set>

#include "../sphericart_amd/csrc/sphx_columns.hpp"
#include "../sphericart_amd/csrc/sphx_plan.hpp"
#include "../sphericart_amd/csrc/sphx_plan_shapes.hpp"

using namespace sphx;

static std::set<size_t> points() {
    std::set<size_t> all;
    for (double n = 1; n < 2e7; n = n * 1.07 + 1) all.insert(static_cast<size_t>(n));
    auto edges = [&](unsigned long long n) {
        for (unsigned long long at : {n - 1, n, n + 1}) {
            if (at >= 1 && at < 20000000ull) all.insert(static_cast<size_t>(at));
        }
    };
    for (const FixedRow& r : kFixedRows) {
        edges(r.points_from);
        edges(r.points_below);
    }
    for (const ShapeRow& r : kShapeRows) {
        edges(r.points_from);
        edges(r.points_below);
    }
    return all;
}

static bool matches(const FixedRow& r, int mode, int elem, int l_max, bool normalized, size_t n) {
    return r.mode == mode && r.elem == elem && l_max >= r.l_from && l_max <= r.l_to && n >= r.points_from && n < r.points_below &&
           (r.harmonics < 0 || r.harmonics == static_cast<int>(normalized));
}

int main() {
    const std::set<size_t> all = points();
    const int lds = 160 * 1024, cus = 256;
    (void)refresh_switches();
    // which rows the calls of a mode, type and l_max come to
    std::set<std::pair<const void*, int>> reached;
    for (int elem : {4, 8}) {
        for (int l_max = 0; l_max <= 64; ++l_max) {
            for (size_t n : all) {
                VjpPlan product;
                ColumnsLaunch columns;
                if (l_max > 6 && make_vjp_plan(n, l_max, elem, lds, cus, &product) == 0 && product.use_lanes &&
                    !vjp_by_columns(n, l_max, elem, lds, cus, product, &columns)) {
                    reached.insert({shape_row(1, elem, l_max, n), l_max});
                }
                for (int mode = 0; mode < 3; ++mode) {
                    for (bool normalized : {false, true}) {
                        Plan plan;
                        if (make_plan(n, l_max, mode, elem, lds, cus, &plan, true, normalized) != 0) continue;
                        const bool fixed = plan.lanes && plan.closed.g.fixed != 0;
                        const FixedRow* row = nullptr;
                        bool another = false; // a row further down names a tile
                        for (const FixedRow& r : kFixedRows) {
                            if (!matches(r, mode, elem, l_max, normalized, n)) continue;
                            if (row == nullptr) row = &r;
                            else if (r.tile != 0) another = true;
                        }
                        if (row != nullptr && (row->tile == 0 ? !fixed && another : fixed)) reached.insert({row, l_max});
                        if (mode == 0 && plan.lanes && !fixed) reached.insert({shape_row(0, elem, l_max, n), l_max});
                        const PriorityRow* raised = priority_row(mode, elem, normalized, l_max);
                        if (raised == nullptr || plan.lanes || plan.closed_only) continue;
                        const unsigned priorities = plan.pairs ? plan.pairs_launch.g.priorities : plan.rec.g.priorities;
                        const unsigned waves = plan.pairs ? plan.pairs_launch.g.sequence_waves : plan.rec.g.sequence_waves;
                        if (priorities == raised->priorities && (raised->sequence_waves == 0 || waves == raised->sequence_waves) &&
                            (priorities != 0 || raised->sequence_waves != 0)) {
                            reached.insert({raised, l_max});
                        }
                    }
                }
            }
        }
    }
    auto report = [&](const char* table, int at, int mode, int elem, int l_from, int l_to, const void* row) {
        for (int l_max = l_from; l_max <= l_to; ++l_max) {
            if (reached.count({row, l_max}) == 0) std::printf("%s %d: %d %d l_max = %d\n", table, at, mode, elem, l_max);
        }
    };
    int at = 0;
    for (const FixedRow& r : kFixedRows) report("kFixedRows", at++, r.mode, r.elem, r.l_from, r.l_to, &r);
    at = 0;
    for (const ShapeRow& r : kShapeRows) report("kShapeRows", at++, r.kind, r.elem, r.l_from, r.l_to, &r);
    at = 0;
    for (const PriorityRow& r : kFlushPriorityRows) report("kFlushPriorityRows", at++, r.mode, r.elem, r.l_from, r.l_to, &r);
    std::printf("done\n");
    return 0;
}
