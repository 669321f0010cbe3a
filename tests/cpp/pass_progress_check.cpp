// The progress records of a handle's passes, with this program in the device's place: reports that arrive
// late, out of the host's sight, or from a pass that was left while its iterations were queued.
// Exit status: number of the failed expectation, 0 if none.
#include "../../naivetrace_amd/csrc/pass_progress.hpp"
#include <cstdio>
using namespace ttgpu;

static int g_checks = 0, g_failed = 0;
static void expect(bool ok, const char *what) {
  ++g_checks;
  if (!ok) {
    printf("%d: %s\n", g_checks, what);
    if (!g_failed) g_failed = g_checks;
  }
}

int main() {
  PassProgress records[2] = {};
  ProgressRecords p;
  p.Attach(records, records);
  auto report = [&](unsigned long long seq, unsigned long long issued, unsigned long long queued) { *p.Device(seq) = {issued, queued, seq}; };
  // A pass of three iterations, its reports in time.
  unsigned long long seq = 0;
  for (int it = 0; it < 3; ++it) {
    seq = p.Next();
    expect(!p.Arrived(seq), "nothing has been reported yet");
    report(seq, 100 + it, 3 - it);
    expect(p.Arrived(seq) && p.Record(seq).issued == 100ull + it && p.Record(seq).queued == 3ull - it, "the iteration's own report");
    if (it > 0) expect(p.Arrived(seq - 1) && p.Record(seq - 1).issued == 99ull + it, "the one before is still there");
  }
  // A pass is left with two iterations queued; their reports come when the next pass has launched its own.
  const unsigned long long left[2] = {p.Next(), p.Next()};
  const unsigned long long first = p.Next(), second = p.Next();
  expect(!p.Arrived(first) && !p.Arrived(second), "the old pass has not reported");
  for (unsigned long long s : left) report(s, 7, 0);
  expect(!p.Arrived(first) && !p.Arrived(second), "a report of the pass that was left is not the new pass's");
  report(first, 8, 5);
  expect(p.Arrived(first) && !p.Arrived(second) && p.Record(first).queued == 5, "the new pass's first report");
  report(second, 8, 0);
  expect(p.Arrived(second) && p.Record(second).issued == 8, "and its second");
  printf("%d checks\n", g_checks);
  return g_failed;
}
