// A short-lived pool of host threads (host code, no GPU types).
#pragma once
#include <thread>
#include <vector>

namespace ccqpool {

// work(0) on the calling thread beside work(1), ..., work(n - 1) on threads of
// their own, all ended on return.  work must not throw, and any of them alone
// must be able to finish the job: a thread that cannot be made (no thread or
// no memory left) is one worker fewer.
template <typename Work>
void run(int n, Work&& work) {
  std::vector<std::thread> pool;
  try {
    pool.reserve((size_t)(n > 1 ? n - 1 : 0));
    for (int w = 1; w < n; ++w) pool.emplace_back([&work, w] { work(w); });
  } catch (...) {
  }
  work(0);
  for (std::thread& t : pool) t.join();
}

}  // namespace ccqpool
