// Planted descriptor offsets that lie inside the operator table but outside the part of it
// that an evaluation reads: the plan's validation has to refuse them.
//   validate_main <ldfile> <hdfile>
#include <cmath>
#include <cstdio>
#include <functional>

#include "planner.hpp"

using namespace ddfmm;

static bool refused(const HostPlan& plan, const std::function<bool(HostPlan&)>& plant, const char* what) {
    HostPlan p = plan;
    if (!plant(p)) {
        std::printf("%s: no such descriptor\n", what);
        return false;
    }
    try {
        validate_plan(p);
    } catch (const std::exception& e) {
        std::printf("%s: %s\n", what, e.what());
        return true;
    }
    std::printf("%s: accepted\n", what);
    return false;
}

int main(int argc, char** argv) {
    if (argc != 3) return 2;
    Mlib lib;
    lib.load(argv[1], argv[2]);
    const int n = 6000;
    const double K = 4.0;
    std::vector<double> pos;
    for (int i = 0; i < n; ++i) {       // spiral points on the sphere of radius 0.47 K
        const double z = 1 - (2 * i + 1.0) / n, s = std::sqrt(1 - z * z), t = 2.399963229728653 * i;
        for (double x : {s * std::cos(t), s * std::sin(t), z}) pos.push_back(0.47 * K * x);
    }
    bool ok = true;
    for (int xlat = 0; xlat < 3; ++xlat)
        for (bool fuse : {false, true}) {
            if (xlat > 0 && !fuse) continue;
            Params q;
            q.K = K;
            q.fuse_solves = fuse;
            q.xlat = xlat;
            HostPlan plan;
            build_plan(q, pos.data(), n, lib, plan, false);
            validate_plan(plan);
            ok &= refused(plan, [](HostPlan& p) {
                for (VTarget& v : p.vtrg) v.tab_off += p.opmat_total - p.opmat_up;
                return !p.vtrg.empty();
            }, "V-list tables in the generated part");
            if (!fuse)
                ok &= refused(plan, [](HostPlan& p) {
                    for (GGroup& g : p.groups)
                        if (g.soff >= 0) {
                            g.soff = p.opmat_total - g.M;
                            return true;
                        }
                    return false;
                }, "row scale in the generated part");
        }
    std::printf(ok ? "all refused\n" : "FAILED\n");
    return ok ? 0 : 1;
}
