// qg_plan_store.hpp — what a handle keeps between calls, safe against a making step that throws: host
// code without HIP, also compiled by the tests.
#pragma once
#include <cstdint>

namespace qg {

// Runs a making step once; a step that throws is run again by the next call.
class MadeOnce {
    bool made_ = false;

public:
    template <class F>
    void operator()(F&& make) {
        if (made_) return;
        make();
        made_ = true;
    }
};

// The last N plans by (precision, batch).  Plan: default-constructible, release() gives back what it
// holds, also half made.  A plan whose making throws leaves its place empty.
template <class Plan, int N>
class PlanStore {
    struct Place {
        bool made = false;
        int prec = 0, batch = 0;
        uint64_t used = 0;
        Plan plan;
    };
    Place places_[N];
    uint64_t uses_ = 0;

public:
    ~PlanStore() {
        for (Place& p : places_) p.plan.release();
    }
    // retire(): called before a plan that may be in use is given back; make(plan)
    template <class Retire, class Make>
    Plan& get(int prec, int batch, Retire&& retire, Make&& make) {
        Place* place = nullptr;
        for (Place& p : places_)
            if (p.made && p.prec == prec && p.batch == batch) place = &p;
        if (!place) {
            place = &places_[0];
            for (Place& p : places_)
                if (p.used < place->used) place = &p;
            if (place->made) {
                retire();
                place->made = false;
                place->used = 0;
            }
            place->plan.release();
            make(place->plan);
            place->made = true;
            place->prec = prec;
            place->batch = batch;
        }
        place->used = ++uses_;
        return place->plan;
    }
};

}  // namespace qg
