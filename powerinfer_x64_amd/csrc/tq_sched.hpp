// tq_sched.hpp -- how a TurboQuant append launch groups its rows (tq_append_kernel,
// turboquant.hip): plain integer arithmetic, apart so that a host test can check it.
#pragma once
#include <stdint.h>

namespace pi {
namespace sched {

struct TqAppendPlan {
    int r;            // tokens per group: consecutive positions of one sequence, aligned to r
    int wpr;          // wavefronts that share a group's coordinates
    long long n_grp;  // groups per (sequence, KV head)
};

// Groups of r aligned positions that n_tok positions from anywhere can touch.
inline long long tq_groups(long long n_tok, int r) { return (n_tok + r - 2) / r + 1; }

// The plan for n_tok tokens of n_seq sequences, head_dim 128 or 256.
//
// Rows per group: as many as leave the chip enough wavefronts (measured, D 128, 8 heads, long
// runs: 8 rows 8.2 us at r 1, 2048 rows 13.8 at r 2 and 16.2 at r 1, 8192 28.4 at r 4 and 32.8
// at r 2, 16 384 44.5 at r 8 and 46.5 at r 4), and no more than the tokens of a sequence are
// worth: a group computes all its r rows, also those that the launch does not cover.  On a full
// chip a group of 1, 2, 4, 8 rows costs 100, 105, 140, 240, so the r of the least groups x cost
// is taken: 1 for 1 or 2 tokens, 2 for 3, 4 for 4 and 8 .. 16, 8 for long runs.  Of 1024
// sequences x 8 heads, D 128, one token took 50 us at r 1 and 119 at r 8, two tokens 93 and 228,
// eight 179 at r 4 and 216 at r 8.
//
// Wavefronts per group: D / 64, shorter chains, until the groups alone fill the chip and reading
// the rows' LDS values in every wavefront costs more.  At r 4: D 128 24.8 us over two wavefronts
// and 23.9 over one at 2048 groups, 33.0 and 30.0 at 3072, 75.0 and 67.2 at 8192; D 256 28.0
// over four, 38.1 over two at 512 groups, 44.8, 40.7 and 66.3 over four, two and one at 1024,
// 78.6, 69.1 and 68.7 at 2048.  At r 8 a lone wavefront takes 95 us (D 256) and a launch few
// rounds of them, so it pays later: D 128 70 us split and 76 not at 4608 groups, 123 and 118 at
// 8320; D 256 130 and 146 at 2080, 252 and 228 at 4608.
inline TqAppendPlan tq_append_plan(long long n_seq, long long n_tok, long long n_kv, int head_dim) {
    constexpr int kCost[4] = {100, 105, 140, 240};
    const long long seqs = n_seq * n_kv, units = seqs * n_tok * (head_dim / 128);
    const int most = units >= 8192 ? 8 : units >= 4096 ? 4 : units >= 2048 ? 2 : 1;
    TqAppendPlan p{1, head_dim / 64, n_tok};
    long long cost = n_tok * kCost[0];
    for (int i = 1; 1 << i <= most; ++i) {
        const long long n = tq_groups(n_tok, 1 << i);
        if (n * kCost[i] < cost) {
            p.r = 1 << i;
            p.n_grp = n;
            cost = n * kCost[i];
        }
    }
    const long long groups = seqs * p.n_grp;
    if (p.r == 8) {
        if (units >= 65536) p.wpr = 1;
    } else if (head_dim == 128) {
        if (groups >= 3072) p.wpr = 1;
    } else {
        if (groups >= 1024) p.wpr = groups >= 2048 ? 1 : 2;
    }
    return p;
}

}  // namespace sched
}  // namespace pi
