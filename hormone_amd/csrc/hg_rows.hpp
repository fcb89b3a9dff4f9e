// hg_rows.hpp -- several threads hand the chunks of a transfer over as they
// arrive.  Host code only.
#pragma once
#include <algorithm>
#include <atomic>
#include <thread>

namespace hg {

// wait(q) returns once chunk q has arrived (chunks arrive in order), false on
// failure; hand(q) hands it over.  Up to `helpers` threads of this call help,
// and are joined before it returns.  They start when the first chunk is there:
// what the transfer itself waits for is not waited for by spinning threads.
// Fewer threads than asked for, or none, only make it slower.
template <class Thread = std::thread, class Wait, class Hand>
bool hand_over_chunks(long nchunk, long helpers, Wait wait, Hand hand) {
  constexpr long MAX = 7;
  if (nchunk <= 0) return true;
  if (!wait(0L)) return false;
  // chunks [0, ready) have arrived; nchunk + 1 tells the helpers to give up
  std::atomic<long> ready{1}, next{0};
  auto help = [&] {
    for (long q; (q = next.fetch_add(1)) < nchunk;) {
      long got;
      while ((got = ready.load(std::memory_order_acquire)) <= q) std::this_thread::yield();
      if (got > nchunk) return;
      hand(q);
    }
  };
  Thread th[MAX];
  long nth = 0;
  try {
    for (; nth < std::min(helpers, MAX); ++nth) th[nth] = Thread(help);
  } catch (...) {  // no thread or no memory to be had
  }
  bool ok = true;
  for (long q = 1; q < nchunk && ok; ++q) {
    ok = wait(q);
    ready.store(ok ? q + 1 : nchunk + 1, std::memory_order_release);
  }
  if (ok) help();
  for (long q = 0; q < nth; ++q) th[q].join();
  return ok;
}

}  // namespace hg
