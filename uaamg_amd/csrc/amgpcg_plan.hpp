// amgpcg_plan.hpp -- sizes of the amgpcg solve's launches and of their partial
// sums (host only; no HIP).
#pragma once
#include <algorithm>

namespace uaamg {

constexpr int AT_X = 32, AT_Y = 16;              // a level's tile (k_ag_down, k_ag_up)
constexpr int AP_X = 64, AP_Y = 16;              // the operator's (k_ag_pmv)
constexpr int AG_TAIL = 64;                      // largest side of the one-workgroup levels

// Every workgroup of the operator and of level 0's down launch adds the
// partials of the launch before it: workgroups times partials, N^4.  Up to
// AG_PARTIALS of them (N = 1024) that costs less than a launch; above, a launch
// of AG_FOLD workgroups folds them to AG_FOLD sums first.
constexpr int AG_PARTIALS = 2048, AG_FOLD = 256;

struct AgPlan {
    int nm, nu;        // partials of p.Ap; of r.r and r.z
    bool fold;
    int sum_m, sum_z;  // how many a consumer adds
    long blocks_m;     // workgroups of the operator (they add sum_z); level 0's down launch has nu
    long doubles;      // all of them
};
inline long ag_partials_room(int N) { return (long)((N + 63) / 64) * ((N + 3) / 4) + 64; }
inline AgPlan ag_plan(int N) {
    AgPlan p{};
    const int my = (N + AP_Y - 1) / AP_Y, ty = (N + AT_Y - 1) / AT_Y;
    const bool tiled = N > AG_TAIL;
    p.nm = (N + AP_X - 1) / AP_X * my;
    p.nu = tiled ? (N + AT_X - 1) / AT_X * ty : std::min(64, (N * N + 255) / 256);
    p.fold = tiled && std::max(p.nm, p.nu) > AG_PARTIALS;
    p.blocks_m = p.nm;
    p.sum_m = p.fold ? AG_FOLD : p.nm;
    p.sum_z = p.fold ? AG_FOLD : (tiled ? p.nu : 1);   // level 0 in the tail: r.z is its one sum
    p.doubles = (long)p.nm + p.nu + (p.fold ? 2 * AG_FOLD : 0);
    return p;
}

}  // namespace uaamg
