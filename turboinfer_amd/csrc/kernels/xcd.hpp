// xcd.hpp -- workgroups of attention heads on the 8 XCDs (plain C++: host, device).
#pragma once

namespace ti {

// `heads` heads of n workgroups each, in a launch of 8 x xcd_per(heads, n): consecutive workgroups go to the XCDs in turn, workgroup i of XCD x
// takes what xcd_work says.  A head's workgroups share an XCD's L2, and every XCD gets as many of the list as the others (8 n heads / 8 rounded
// up): heads that divide 8 are shared by 8 / heads XCDs, whose workgroups alternate (a head's first ones have the longest chains); any other
// number of heads is cut into 8 equal runs of the (head, workgroup) list.
constexpr int xcd_per(int heads, int n) { return 8 % heads == 0 ? (n + 8 / heads - 1) / (8 / heads) : (int)(((long)heads * n + 7) / 8); }

struct XcdWork {
  int head, j;   // (head -1: nothing)
};
constexpr XcdWork xcd_work(int heads, int n, int x, int i) {
  if (8 % heads == 0) {
    const int share = 8 / heads, j = i * share + x % share;
    return {j < n ? x / share : -1, j};
  }
  const int per = xcd_per(heads, n), id = x * per + i;
  return {i < per && id < heads * n ? id / n : -1, id % n};
}

}  // namespace ti
