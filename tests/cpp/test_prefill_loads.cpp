// Host walk of the direct loads and waits of prefill_fa_kernel's tile loop (prefill.hip), with the
// counts it takes from prefill_loads.hpp: before the barrier of step t every wavefront's loads of
// unit t + 1 must have arrived, when loads complete in order and its wait leaves vmcnt of them in
// flight, and the units after it are the loads left.  Exit status 0 = every wait is right.
#include "prefill_loads.hpp"

#include <algorithm>
#include <cstdio>
#include <deque>

namespace {

int failures = 0;

template <int D, bool PG>
void walk(int nloc) {
    typedef pi::PrefillLoads<D, PG> L;
    for (int wave = 0; wave < L::NW; ++wave) {
        if (PG && wave >= L::NW / L::LPD) continue;  // issues no loads
        std::deque<int> flight;                      // the unit of every load in flight, oldest first
        auto issue = [&](int u) {
            for (int ps = 0; ps < L::LPD; ++ps) {
                const int wv = wave + ps * (L::NW / L::LPD);
                for (int i = wv; i < L::K_INSTR; i += L::NW) flight.push_back(u);
                if (u >= 1)
                    for (int j = 0; j < L::VJ; ++j) flight.push_back(u);
            }
        };
        issue(0);
        if (nloc >= 1) issue(1);
        flight.clear();  // all waited for before the loop
        if (2 <= nloc) issue(2);
        for (int t = 0; t < nloc; ++t) {
            if (t + 3 <= nloc) issue(t + 3);
            const int ahead = std::min(2, std::max(0, nloc - (t + 1)));
            const size_t left = (size_t)ahead * L::unit_loads(wave);
            while (flight.size() > left) flight.pop_front();
            const bool late = !flight.empty() && flight.front() <= t + 1;
            const bool early = flight.size() < left;  // vmcnt above the loads in flight
            if ((late || early) && failures++ < 20)
                std::printf("FAIL D %d %s wave %d, %d tiles, step %d: %s\n", D, PG ? "paged" : "rows", wave, nloc, t,
                            late ? "unit t + 1 is still in flight at the barrier" : "the wait allows more loads than there are");
        }
    }
}

}  // namespace

int main() {
    for (int nloc = 1; nloc <= 12; ++nloc) {
        walk<64, false>(nloc);
        walk<64, true>(nloc);
        walk<128, false>(nloc);
        walk<128, true>(nloc);
    }
    std::printf("%d failures\n", failures);
    return failures != 0;
}
