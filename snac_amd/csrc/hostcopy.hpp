// Copies between a field's rows on the device and a contiguous host array.
#pragma once
#include "common.hpp"

namespace snac {

// A context's staging memory for field uploads and downloads: pinned chunks,
// allocated at the first copy (as many as the largest copy so far can use,
// at most 16 MiB) and freed with the context.
class HostCopy {
public:
  ~HostCopy() { release(); }
  // rows of w doubles, `pitch` doubles apart on the device and contiguous on
  // the host; returns when the copy is complete
  void run(int device, hipStream_t st, double *dev, long pitch, long w, long rows, double *to_host,
           const double *from_host);
  void release();

private:
  static constexpr int SLOTS = 16;          // two per copying thread
  static constexpr long CHUNK = 1L << 17;   // doubles per slot (1 MiB)
  double *slot_[SLOTS] = {};
  long cap_[SLOTS] = {};
  hipEvent_t ev_[SLOTS] = {};
  void need(int slot, long n);
};

}  // namespace snac
