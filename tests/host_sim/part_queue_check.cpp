// Threads that take parts of a document as these arrive (csrc/part_queue.h), without a GPU: the parts come from a
// thread that sleeps between them.
#include <sys/resource.h>
#include <time.h>

#include <vector>

#include "../../kineto_amd/csrc/part_queue.h"

namespace {
double seconds() { timespec t; clock_gettime(CLOCK_MONOTONIC, &t); return (double)t.tv_sec + 1e-9 * (double)t.tv_nsec; }
double cpu_seconds() {
  rusage u;
  getrusage(RUSAGE_SELF, &u);
  return (double)(u.ru_utime.tv_sec + u.ru_stime.tv_sec) + 1e-6 * (double)(u.ru_utime.tv_usec + u.ru_stime.tv_usec);
}
}  // namespace

extern "C" {
/* n_parts parts, gap_us apart (0: as fast as may be), of which arrive_parts come before the rest is given up; n_threads
 * take them.  taken[part] is how often each was taken.  Wall-clock and processor seconds of all of it. */
void ktjsim_part_queue(uint64_t n_parts, uint64_t arrive_parts, unsigned n_threads, unsigned gap_us, uint32_t* taken, double* wall, double* cpu) {
  ktj::PartQueue queue(n_parts);
  const double w0 = seconds(), c0 = cpu_seconds();
  std::vector<std::thread> threads;
  for (unsigned t = 0; t < n_threads; ++t)
    threads.emplace_back([&] {
      for (uint64_t c; queue.take(&c);) __atomic_fetch_add(&taken[c], 1u, __ATOMIC_RELAXED);
    });
  for (uint64_t c = 0; c < arrive_parts; ++c) {
    if (gap_us) std::this_thread::sleep_for(std::chrono::microseconds(gap_us));
    queue.arrive();
  }
  if (arrive_parts < n_parts) queue.give_up();
  for (auto& t : threads) t.join();
  *wall = seconds() - w0;
  *cpu = cpu_seconds() - c0;
}
}
