// Parts of the copies between host and device that need no GPU.
#pragma once

#include <thread>

namespace dn {

// work(0) ... work(n - 1), each on a thread of its own, work(0) on the caller's.  Where no thread can be made
// (`spawn` throws) the shares that are left run on the caller's thread, one after the other.
template <class Work, class Spawn>
void run_shares(int n, Work&& work, Spawn&& spawn) {
  constexpr int MOST = 16;
  std::thread helpers[MOST];
  int made = 1;
  try {
    for (; made < n && made < MOST; made++) helpers[made] = spawn([&work, t = made] { work(t); });
  } catch (...) {
  }
  work(0);
  for (int t = made; t < n; t++) work(t);
  for (int t = 1; t < made; t++) helpers[t].join();
}

}  // namespace dn
