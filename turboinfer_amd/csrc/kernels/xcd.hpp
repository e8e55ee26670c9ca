// xcd.hpp -- workgroups of attention heads on the 8 XCDs (plain C++: host, device).
#pragma once

namespace ti {

// `heads` heads of n workgroups each, in a launch of 8 x per: consecutive workgroups go to the XCDs in turn, workgroup i of XCD x takes what
// xcd_work says.  A head's workgroups share an XCD's L2, and every XCD gets as many of the list as the others (heads n / 8, rounded up): heads
// that divide 8 are shared by 8 / heads XCDs, whose workgroups alternate (a head's first ones have the longest chains); any other number
// of heads is cut into 8 equal runs of the (head, workgroup) list.  us, head_dim 128, a head an XCD (heads x, x + 8, ..) -> this: 40 heads on 10,
// 200 rows 14.7 -> 8.5 (spread over all XCDs in turn 8.4), 1000 65.0 -> 50.9 (56.3); 40 on 5, 400 rows 20.8 -> 12.4 (12.6); latent, 12
// heads, 1300 rows 44.9 -> 28.0.
//
// Workgroups of `share` XCDs alternate in runs of `run` items of the list.  (Without branches and divisions: in front of a short launch's first
// loads they took 0.3 us of 8.)
struct XcdDeal {
  int list, n, per, run, log_share;
  unsigned inv;   // (2^32 - 1) / n
};
struct XcdWork {
  int head, j;   // (head -1: nothing)
};
constexpr int kXcdRows = 32768;   // of the launch's y: more workgroups an XCD go to z
constexpr XcdDeal xcd_deal(int heads, int n) {
  const int log_share = heads == 4 ? 1 : heads == 2 ? 2 : heads == 1 ? 3 : 0, run = log_share ? n : (int)(((long)heads * n + 7) / 8);
  return {heads * n, n, (run + (1 << log_share) - 1) >> log_share, run, log_share, 0xffffffffu / (unsigned)n};
}
constexpr XcdWork xcd_work(const XcdDeal& d, int x, int i) {
  const int first = (x >> d.log_share) * d.run, id = first + (x & ((1 << d.log_share) - 1)) + (i << d.log_share);
  const int end = first + d.run < d.list ? first + d.run : d.list;
  int head = (int)((unsigned long long)(unsigned)id * d.inv >> 32), j = id - head * d.n;   // (at most one too small)
  if (j >= d.n) {
    ++head;
    j -= d.n;
  }
  return {id < end ? head : -1, j};
}

}  // namespace ti
