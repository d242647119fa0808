// Host driver of qg_plan_store.hpp: plans that count what they hold, and making steps that throw at a
// chosen point.  Exits 0 where every check holds, and names the first that does not.
#include <cstdio>
#include <cstdlib>
#include "../../qumasun_amd/csrc/qg_plan_store.hpp"

static int held = 0;
struct Plan {
    int fwd = 0, inv = 0;
    void release() {
        held -= (fwd != 0) + (inv != 0);
        fwd = inv = 0;
    }
};
#define CHECK(c)                                        \
    if (!(c)) {                                         \
        std::printf("line %d: %s\n", __LINE__, #c);     \
        return 1;                                       \
    }

int main() {
    // a making step that throws is run again
    qg::MadeOnce once;
    int runs = 0;
    for (int k = 0; k < 4; ++k) {
        try {
            once([&] {
                if (++runs < 3) throw 1;
            });
        } catch (int) {
        }
    }
    CHECK(runs == 3);

    int made = 0, retired = 0;
    {
        qg::PlanStore<Plan, 3> store;
        auto retire = [&] { ++retired; };
        // fail: 0 never, 1 before the first part, 2 between the parts, 3 after both
        auto get = [&](int prec, int batch, int fail = 0) -> Plan* {
            try {
                return &store.get(prec, batch, retire, [&](Plan& p) {
                    if (fail == 1) throw 1;
                    p.fwd = 1000 * prec + batch, ++held;
                    if (fail == 2) throw 1;
                    p.inv = p.fwd, ++held;
                    if (fail == 3) throw 1;
                    ++made;
                });
            } catch (int) {
                return nullptr;
            }
        };
        for (int fail = 1; fail <= 3; ++fail) {
            CHECK(!get(0, 5, fail));
            Plan* p = get(0, 5 + fail);
            CHECK(p && p->fwd == 5 + fail && p->inv == p->fwd);
            CHECK(!get(1, 5 + fail, fail));                  // another precision, not the plan of this one
            CHECK((p = get(0, 5 + fail)) && p->fwd == 5 + fail);
        }
        CHECK(made >= 3 && held <= 6);
        // the three last used stay, the oldest goes
        made = retired = 0;
        get(2, 1), get(2, 2), get(2, 3), get(2, 1), get(2, 4);
        CHECK(retired >= 1);
        made = 0;
        get(2, 1), get(2, 3), get(2, 4);
        CHECK(made == 0);
        get(2, 2);
        CHECK(made == 1);
        // a plan that replaces an old one and fails leaves neither behind
        CHECK(!get(3, 9, 3));
        CHECK(get(3, 9)->fwd == 3009);
        CHECK(held == 6);
    }
    CHECK(held == 0);
    std::printf("ok\n");
    return 0;
}
