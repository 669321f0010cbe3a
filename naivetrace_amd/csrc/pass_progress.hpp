// How a pass's iterations report to the host: records in page-locked memory that the device writes.
#pragma once
#include <algorithm>
#include <cstdint>

namespace ttgpu {

// Progress record of an iteration, written by the device: camera paths issued, work queued for the
// next iteration, and the iteration's number (written last).
struct PassProgress {
  unsigned long long issued, queued, seq;
};

// The host's side of a handle's two records (even and odd iterations).  Iterations are numbered through
// the handle's whole life: a report of a pass that was left by an exception, arriving after the next
// pass has begun, is none that the next pass waits for.
class ProgressRecords {
 public:
  // `records`: two, in host memory; `device`: their device address.
  void Attach(PassProgress *records, PassProgress *device) {
    host_ = records;
    device_ = device;
  }
  // Number of the iteration about to be launched.
  unsigned long long Next() { return ++last_; }
  PassProgress *Device(unsigned long long seq) const { return device_ + (seq & 1); }
  const PassProgress &Record(unsigned long long seq) const { return host_[seq & 1]; }
  // At most one further iteration may have been launched.
  bool Arrived(unsigned long long seq) const { return __atomic_load_n(&host_[seq & 1].seq, __ATOMIC_ACQUIRE) == seq; }

 private:
  PassProgress *host_ = nullptr, *device_ = nullptr;
  unsigned long long last_ = 0;
};

}  // namespace ttgpu
