// The grouping of TurboQuant append launches (powerinfer_x64_amd/csrc/tq_sched.hpp) on the host.
// Without arguments: checks every plan of a range of launches.  With "n_seq n_tok n_kv head_dim":
// prints that launch's "r wpr", for the tests that must know which kernel a launch picks.
#include "tq_sched.hpp"

#include <cstdio>
#include <cstdlib>
#include <initializer_list>

using namespace pi::sched;

int main(int argc, char** argv) {
    if (argc == 5) {
        const TqAppendPlan p = tq_append_plan(std::atoll(argv[1]), std::atoll(argv[2]), std::atoll(argv[3]),
                                              std::atoi(argv[4]));
        std::printf("%d %d\n", p.r, p.wpr);
        return 0;
    }
    int failures = 0;
    auto fail = [&](const char* what, long long s, long long n, long long h, int d, const TqAppendPlan& p) {
        if (failures++ < 20)
            std::printf("FAIL %s: n_seq %lld n_tok %lld heads %lld D %d: r %d wpr %d n_grp %lld\n", what, s, n, h, d,
                        p.r, p.wpr, p.n_grp);
    };
    const long long seqs[] = {1, 2, 32, 256, 1024, 4096, 65536}, heads[] = {1, 2, 8, 32};
    for (int d : {128, 256})
        for (long long s : seqs)
            for (long long h : heads)
                for (long long n = 1; n <= 600; n += n < 70 ? 1 : 53) {
                    const TqAppendPlan p = tq_append_plan(s, n, h, d);
                    if (p.r != 1 && p.r != 2 && p.r != 4 && p.r != 8) fail("rows", s, n, h, d, p);
                    // the kernels that exist
                    if (p.wpr != 1 && p.wpr != d / 64 && !(p.wpr == 2 && p.r < 8)) fail("wavefronts", s, n, h, d, p);
                    // a group computes all its rows: at most twice the launch's own
                    if (p.n_grp * p.r > 2 * n) fail("rows computed", s, n, h, d, p);
                    // the groups cover the tokens from any start, and none is spare at the worst one
                    long long most = 0;
                    for (long long at = 0; at < 16; ++at) {
                        const long long used = (at + n - 1) / p.r - at / p.r + 1;
                        most = used > most ? used : most;
                    }
                    if (most != p.n_grp) fail("groups", s, n, h, d, p);
                }
    std::printf("%d failures\n", failures);
    return failures != 0;
}
