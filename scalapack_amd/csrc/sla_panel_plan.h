// sla_panel_plan.h -- how a panel leaf (panel.hip) of m rows and wa columns is cut
// into workgroups, and where they run.  Host code only.
#pragma once

#include <algorithm>

namespace sla {

constexpr int LEAF_GMAX = 128;         // workgroups per leaf launch at most
constexpr int XCDS = 8, XCD_CUS = 32;  // the dies of the GPU and the CUs of one

// Where the workgroups go: dealt over all XCDs, all on one, or all on one with a
// second launch, dealt over all, that does the work if the first gave way.
enum LeafPlace { LEAF_SPREAD, LEAF_ONE_XCD, LEAF_ONE_XCD_YIELDS };

struct LeafPlan {
    int values;  // matrix elements a thread holds: 16 or 32 take at most 128 registers, 64 up to 256
    int waves;   // of a workgroup
    int wgs;     // workgroups (above LEAF_GMAX: the leaf is too tall)
    LeafPlace place;
};

// Registers per row and lane by the leaf's width (a row lies in four lanes).
constexpr int leaf_nc(int wa) { return wa <= 8 ? 2 : wa <= 16 ? 4 : 8; }
// Elements a thread holds in the smaller kinds.
constexpr int leaf_values(int nc) { return nc == 2 ? 16 : 32; }
// Kinds (by registers per row and lane, threads) that may be planned to give way.
constexpr bool leaf_may_yield(int nc, int threads) { return nc == 8 && threads == 512; }
// Quarters of a CU that a workgroup's registers take.
constexpr int leaf_quarters(const LeafPlan &p) { return (p.values == 64 ? 2 : 1) * (p.waves > 4 ? 2 : 1); }

// panel_wgs: the workgroups that the caller prefers at most; four times as many of
// the smallest kind beside an update and for narrow leaves.  beside: a long trailing update runs on another stream meanwhile.  xcds: the GPU has all
// its XCDs' CUs.
inline LeafPlan leaf_plan(int m, int wa, int panel_wgs, bool beside, bool xcds)
{
    const int nc = leaf_nc(wa), v = leaf_values(nc);
    auto grid = [&](int values, int waves) {
        const int rows = 16 * (values / nc) * waves;
        return (m + rows - 1) / rows;
    };
    const int g1 = grid(v, 4), g2 = grid(v, 8), g3 = grid(64, 8);
    // One workgroup while it holds the leaf: 78 us at m = 1000 and without the
    // other streams' kernels in the way of an exchange.  (16 waves of 32 values
    // instead of 8 of 64: 80 us; a SIMD's four waves wait for each other.)
    if (g2 == 1) return {v, grid(v, 1), 1, LEAF_SPREAD};
    if (nc == 8 && g3 == 1) return {64, grid(64, 1), 1, LEAF_SPREAD};
    // Then as many as one XCD runs, of the smallest kind: 82 us at m = 8192 with
    // four waves.  Beside a long trailing update only those find room, so there
    // they go on, across the XCDs: m = 16384 alone 139 us, with eight waves 95 us,
    // but these wait for the end of the update.  Leaves of at most 16 columns go on
    // there always: their steps are short, 64 values of so few columns are many rows
    // a quad, and those come one after another (8 columns, m = 2000: one workgroup
    // 55 us, eight 25; m = 50000: 13 workgroups 117 us, 98 of the smallest kind 45; 16
    // columns: 66, 48; 100, 83).
    //
    // Workgroups that wait for one another have to run together, whatever else runs.
    // The smallest kind takes a quarter of a CU, so an XCD holds four leaves of it
    // at once: as many as HIP's four hardware queues run of a process's handles.
    // The larger kinds take half a CU and a whole one.  On one XCD two leaves
    // of theirs could keep each other out, each with a part of its workgroups
    // running, so these give way (keep_waiting in panel.hip): a launch over all
    // XCDs, where eight of them find room, follows and does the work instead.
    auto tall = [&](int g) { return xcds && wa > 1 && g <= XCD_CUS ? LEAF_ONE_XCD_YIELDS : LEAF_SPREAD; };
    if (g1 <= (beside || nc < 8 ? std::min(4 * panel_wgs, LEAF_GMAX) : panel_wgs))
        return {v, 4, g1, xcds && g1 <= XCD_CUS ? LEAF_ONE_XCD : LEAF_SPREAD};
    if (nc == 8 && g2 <= panel_wgs) return {v, 8, g2, tall(g2)};
    if (nc == 8 && g3 <= panel_wgs) return {64, 8, g3, tall(g3)};
    // with more than the caller prefers, the fewest, on one XCD
    if (nc == 8 && g3 <= XCD_CUS) return {64, 8, g3, tall(g3)};
    // Over the XCDs the middle kind is the faster one (32 columns, m = 65536: 174 us
    // against 179 with half as many of the largest kind; 16 columns, 131072: 99, 115)
    if (g2 <= LEAF_GMAX) return {v, 8, g2, LEAF_SPREAD};
    return {64, 8, g3, LEAF_SPREAD};
}

}  // namespace sla
