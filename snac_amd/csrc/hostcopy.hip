// Field uploads and downloads.  A field's rows are padded on the device and
// contiguous on the host, and the host array is ordinary pageable memory.  A
// pitched hipMemcpy to pageable memory moves it row by row (7 us a row down,
// 9 us up: 0.56 GB/s at 514 doubles a row, 0.08 GB/s at 66).  Here a kernel
// packs chunks of rows straight into pinned host memory, and host threads
// move the chunks to the caller's array while the next ones are packed: a
// 70 MB field comes down in 2.3 ms (30 GB/s) instead of 122 ms, one of 37 KB
// in 0.03 ms instead of 7.8 ms.
#include "hostcopy.hpp"

#include <climits>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace snac {
namespace {

// The packed elements [0, n) of a chunk that starts at element c0 of a row
// whose device address is d; bound by the link to the host, so 8-byte
// accesses (rows start 8 bytes off a 128-byte line) are as fast as wider ones.
template <bool UP>
__global__ __launch_bounds__(256) void k_pack_rows(double *__restrict__ d, long pitch, unsigned w, unsigned c0,
                                                   unsigned n, double *__restrict__ pin) {
  for (unsigned t = blockIdx.x * 256 + threadIdx.x; t < n; t += gridDim.x * 256) {
    const unsigned e = c0 + t, row = e / w;
    double *p = d + row * pitch + (e - row * w);
    if (UP) *p = pin[t];
    else pin[t] = *p;
  }
}

}  // namespace

void HostCopy::need(int s, long n) {
  if (cap_[s] < n) {
    if (slot_[s]) (void)hipHostFree(slot_[s]);
    slot_[s] = nullptr;
    cap_[s] = 0;
    SNAC_HIP(hipHostMalloc((void **)&slot_[s], n * sizeof(double), hipHostMallocDefault));
    cap_[s] = n;
  }
  if (!ev_[s]) SNAC_HIP(hipEventCreateWithFlags(&ev_[s], hipEventDisableTiming));
}

void HostCopy::release() {
  for (int s = 0; s < SLOTS; s++) {
    if (slot_[s]) (void)hipHostFree(slot_[s]);
    if (ev_[s]) (void)hipEventDestroy(ev_[s]);
    slot_[s] = nullptr;
    ev_[s] = nullptr;
    cap_[s] = 0;
  }
}

void HostCopy::run(int device, hipStream_t st, double *dev, long pitch, long w, long rows, double *to_host,
                   const double *from_host) {
  if (!to_host && !from_host) throw std::runtime_error("null host array");
  if (w <= 0 || rows <= 0) return;
  if (w > INT_MAX) throw std::runtime_error("field copy: row too long");  // k_pack_rows counts within w + CHUNK in 32 bits
  const long n = w * rows, nchunk = (n + CHUNK - 1) / CHUNK;
  // one thread keeps up with the link while the caller's pages are mapped; a
  // fresh array's page faults take about 0.1 ms per MiB and thread, so from
  // 4 MiB on up to eight threads share them (their start costs ~0.1 ms)
  int nt = 1;
  if (nchunk >= 4) {
    const unsigned hw = std::thread::hardware_concurrency();
    nt = (int)std::min<long>({SLOTS / 2, (nchunk + 1) / 2, hw > 0 ? (long)hw : 1L});
  }
  for (int s = 0; s < 2 * nt && s < nchunk; s++) need(s, std::min(n, CHUNK));
  std::mutex mu;
  std::exception_ptr err;
  // thread t copies chunks t, t + nt, ... through its two slots
  auto work = [&](int t) {
    try {
      if (t > 0) SNAC_HIP(hipSetDevice(device));
      long pend[2] = {-1, -1};
      auto len = [&](long c) { return std::min(CHUNK, n - c * CHUNK); };
      auto pack = [&](long c, int s) {
        const long e0 = c * CHUNK, m = len(c);
        double *d = dev + (e0 / w) * pitch;
        const unsigned c0 = (unsigned)(e0 % w);
        const dim3 g((unsigned)std::min<long>((m + 255) / 256, 256));
        if (from_host) hipLaunchKernelGGL(k_pack_rows<true>, g, dim3(256), 0, st, d, pitch, (unsigned)w, c0, (unsigned)m, slot_[s]);
        else hipLaunchKernelGGL(k_pack_rows<false>, g, dim3(256), 0, st, d, pitch, (unsigned)w, c0, (unsigned)m, slot_[s]);
        SNAC_HIP(hipGetLastError());
        SNAC_HIP(hipEventRecord(ev_[s], st));
      };
      auto drain = [&](int q) {
        if (pend[q] < 0) return;
        SNAC_HIP(hipEventSynchronize(ev_[2 * t + q]));
        if (to_host) std::memcpy(to_host + pend[q] * CHUNK, slot_[2 * t + q], len(pend[q]) * sizeof(double));
        pend[q] = -1;
      };
      int q = 0;
      for (long c = t; c < nchunk; c += nt, q ^= 1) {
        drain(q);
        if (from_host) std::memcpy(slot_[2 * t + q], from_host + c * CHUNK, len(c) * sizeof(double));
        pack(c, 2 * t + q);
        pend[q] = c;
      }
      drain(q);
      drain(q ^ 1);
    } catch (...) {
      std::lock_guard<std::mutex> lk(mu);
      if (!err) err = std::current_exception();
    }
  };
  std::vector<std::thread> th;
  try {
    for (int t = 1; t < nt; t++) th.emplace_back(work, t);
  } catch (...) {  // fewer threads than asked for: their chunks are copied here
  }
  const int started = (int)th.size();
  work(0);
  for (int t = started + 1; t < nt; t++) work(t);
  for (auto &x : th) x.join();
  if (err) {
    (void)hipStreamSynchronize(st);  // no kernel of this copy outlives it
    std::rethrow_exception(err);
  }
}

}  // namespace snac
