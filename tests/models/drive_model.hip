// Host model of the phase driver (gb_drive_loop): a device that runs launches
// behind the host and reports the phases it has begun in several ways.
#include <cstdio>
#include <cstdlib>
#include <deque>

#include "gb_internal.hpp"

gb_status gb_fail(gb_status s, const char *, ...) { return s; }
uint64_t gb_next_graph_uid() { return 0; }
void gb_dfree(void *) {}
gb_status gb_dmalloc(void **, size_t) { return GB_ERR_NOMEM; }

// A stream whose launches run only while the host waits (lazy) or at once.
struct Device {
  GbProgress rec{};
  std::deque<uint32_t> queue;
  uint32_t last;    // the phase that reports the loop done
  uint32_t report;  // reports every report-th phase; 0: none
  bool lazy;
  uint32_t ran = 0, most = 0;
  void run_one() {
    const uint32_t k = queue.front();
    queue.pop_front();
    if (k != ran++) {
      std::printf("phase %u out of order\n", k);
      std::exit(1);
    }
    if (k >= last)
      rec.done = 1;
    else if (report && k % report == report - 1)
      rec.started = k + 1;
  }
  hipError_t launch(uint32_t k) {
    queue.push_back(k);
    most = queue.size() > most ? (uint32_t)queue.size() : most;
    if (!lazy) run_one();
    return hipSuccess;
  }
  // one phase per look, then dry
  hipError_t query() {
    if (queue.empty()) return hipSuccess;
    run_one();
    return hipErrorNotReady;
  }
};

static int bad = 0;
static void check(const char *what, uint32_t first, uint32_t last, uint32_t report, bool lazy,
                  uint32_t ahead, gb_status want) {
  Device d{};
  d.rec.started = first;
  d.last = last;
  d.report = report;
  d.lazy = lazy;
  const gb_status s = gb_drive_loop(
      &d.rec, ahead, [&](uint32_t k) { return d.launch(k); }, [&]() { return d.query(); });
  // a record that starts ahead admits that many more
  const bool ok = s == want && (want != GB_OK || d.ran > last) && d.most <= ahead + first;
  if (!ok) {
    std::printf("%s: status %d, %u phases run, %u queued at most\n", what, (int)s, d.ran, d.most);
    bad = 1;
  }
}

int main() {
  for (uint32_t ahead : {2u, 6u, 8u})
    for (uint32_t last : {0u, 1u, 2u, 5u, 6u, 7u, 40u})
      for (int lazy = 0; lazy < 2; lazy++) {
        check("every phase", 0, last, 1, lazy, ahead, GB_OK);
        // a record one phase ahead of the host before its first launch
        check("ahead", 1, last, 1, lazy, ahead, GB_OK);
        if (ahead >= 3) check("every third phase", 0, last, 3, lazy, ahead, GB_OK);
      }
  // a device that reports nothing: an error, once the stream is dry
  check("silent", 0, 100, 0, true, 4, GB_ERR_HIP);
  check("silent", 0, 100, 0, false, 4, GB_ERR_HIP);
  if (!bad) std::printf("ok\n");
  return bad;
}
