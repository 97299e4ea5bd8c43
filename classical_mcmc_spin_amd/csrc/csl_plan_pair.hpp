// csl_plan_pair.hpp — two library plans kept for the shape they were made for
// (host side, no HIP).
#pragma once

namespace cslh {

// Plans a and b of shape `key`.  They are kept while the shapes asked for stay
// the same; a failure while making them leaves none, so that what was made for
// one shape never answers for another.
template <class Plan, class Key, void (*Destroy)(Plan)>
class PlanPair {
public:
    Plan a{}, b{};

    PlanPair() = default;
    PlanPair(const PlanPair&) = delete;
    PlanPair& operator=(const PlanPair&) = delete;
    ~PlanPair() { drop(); }

    void drop() {
        if (a) Destroy(a);
        if (b) Destroy(b);
        a = b = Plan{};
        made_ = false;
    }
    // make(a, b) fills both or throws.
    template <class Make>
    void use(const Key& key, Make&& make) {
        if (made_ && key_ == key) return;
        drop();
        try {
            make(a, b);
        } catch (...) {
            drop();
            throw;
        }
        key_ = key;
        made_ = true;
    }

private:
    Key key_{};
    bool made_ = false;
};

}  // namespace cslh
