// Copies between the caller's (pageable) host arrays and the device.
//
// A copy of pageable memory goes through the runtime's own staging: 0.5 MB takes 210 µs,
// 2 MB down 810 µs, 4 MB down 220 µs (17 GB/s), where the same bytes take 18, 44 and
// 76 µs from pinned memory (55 GB/s) and a host copy another 4, 25 and 50 µs.  So the
// library keeps its own pinned staging: a copy is cut into chunks, up to kSlots of them
// in flight, and the host side of one chunk runs while the next ones are on the link.
//
// A staging buffer belongs to one call at a time (HostCopy acquires and returns it).  Idle
// buffers are kept in a process-wide list of at most kMaxIdle (kMaxIdle x 4 MB pinned), and
// of kKeepIdle once no context is left, which is what one call takes at most: so a context of
// a single assembly does not pay for pinning; the list holds no device
// state, any thread and any device's stream may take from it, and a buffer goes back
// only after the copies that use it have finished.  Calls beyond kMaxIdle at once pin
// their own buffer and free it.  Where pinning is refused the runtime's own copies take over.
#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "gh_internal.h"

namespace gh {
namespace {

constexpr size_t kChunk = size_t(1) << 20;
constexpr int kSlots = 4;
constexpr size_t kMaxIdle = 8, kKeepIdle = 2, kBytes = kSlots * kChunk + 64;  // the slots, a word

std::mutex g_mu;
std::vector<char *> g_idle;  // kBytes each
int g_contexts = 0;

// An idle buffer or a new one; null when pinning is refused.
char *take_buffer() {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (!g_idle.empty()) {
      char *b = g_idle.back();
      g_idle.pop_back();
      return b;
    }
  }
  void *b = nullptr;
  if (hipHostMalloc(&b, kBytes, hipHostMallocCoherent | hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();  // else the next call would report it
    return nullptr;
  }
  return static_cast<char *>(b);
}

}  // namespace

void host_copy_context(bool opened) {
  std::lock_guard<std::mutex> lock(g_mu);
  g_contexts += opened ? 1 : -1;
  for (; g_contexts == 0 && g_idle.size() > kKeepIdle; g_idle.pop_back())
    (void)hipHostFree(g_idle.back());
}

HostCopy::HostCopy(Ctx &c, bool direct) : s_(c.stream) {
  if (direct || !c.pinned) return;
  ev_ = c.copy_events();
  buf_ = take_buffer();
}

HostCopy::~HostCopy() {
  if (busy_) (void)hipStreamSynchronize(s_);  // an error path: copies may be in flight
  if (!buf_) return;
  try {
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_idle.size() < kMaxIdle) {
      g_idle.push_back(buf_);
      return;
    }
  } catch (const std::bad_alloc &) {
  }
  (void)hipHostFree(buf_);
}

void HostCopy::wait_slot(int k) {
  if (used_[k]) GH_CHECK_HIP(hipEventSynchronize(ev_[k]));
  used_[k] = false;
}

uint64_t *HostCopy::word() const {
  return buf_ ? reinterpret_cast<uint64_t *>(buf_ + kSlots * kChunk) : nullptr;
}

void HostCopy::up(void *dev, const void *host, size_t bytes) {
  if (!buf_) {
    busy_ = true;
    if (bytes) GH_CHECK_HIP(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s_));
    return;
  }
  for (size_t o = 0; o < bytes; o += kChunk) {
    const size_t n = std::min(kChunk, bytes - o);
    const int k = next_;
    next_ = (next_ + 1) % kSlots;
    wait_slot(k);
    std::memcpy(buf_ + k * kChunk, (const char *)host + o, n);
    busy_ = true;
    GH_CHECK_HIP(hipMemcpyAsync((char *)dev + o, buf_ + k * kChunk, n, hipMemcpyHostToDevice, s_));
    GH_CHECK_HIP(hipEventRecord(ev_[k], s_));
    used_[k] = true;
  }
}

void HostCopy::down_chunks(const void *dev, size_t bytes, size_t unit,
                           const std::function<void(const char *, size_t, size_t)> &take) {
  const size_t chunk = kChunk / unit * unit;
  size_t sent = 0, got = 0;
  int first = next_, pending = 0;
  while (got < bytes) {
    while (sent < bytes && pending < kSlots) {
      const size_t n = std::min(chunk, bytes - sent);
      wait_slot(next_);
      busy_ = true;
      GH_CHECK_HIP(hipMemcpyAsync(buf_ + next_ * kChunk, (const char *)dev + sent, n,
                                  hipMemcpyDeviceToHost, s_));
      GH_CHECK_HIP(hipEventRecord(ev_[next_], s_));
      used_[next_] = true;
      next_ = (next_ + 1) % kSlots;
      sent += n;
      ++pending;
    }
    const size_t n = std::min(chunk, bytes - got);
    wait_slot(first);
    take(buf_ + first * kChunk, got, n);
    first = (first + 1) % kSlots;
    got += n;
    --pending;
  }
}

void HostCopy::down(void *host, const void *dev, size_t bytes) {
  if (!buf_) {
    if (bytes) GH_CHECK_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s_));
    GH_CHECK_HIP(hipStreamSynchronize(s_));
    return;
  }
  down_chunks(dev, bytes, 1, [&](const char *src, size_t at, size_t n) {
    std::memcpy((char *)host + at, src, n);
  });
}

void HostCopy::down_ids(int64_t *host, const int32_t *dev, size_t count) {
  auto widen = [&](const char *src, size_t at, size_t n) {
    const int32_t *in = (const int32_t *)src;
    int64_t *out = host + at / sizeof(int32_t);
    for (size_t k = 0; k < n / sizeof(int32_t); ++k) out[k] = int64_t(in[k]) + 1;
  };
  if (!buf_) {
    std::vector<int32_t> ids(count);
    down(ids.data(), dev, count * sizeof(int32_t));
    widen((const char *)ids.data(), 0, count * sizeof(int32_t));
    return;
  }
  down_chunks(dev, count * sizeof(int32_t), sizeof(int32_t), widen);
}

void HostCopy::finish() {
  GH_CHECK_HIP(hipStreamSynchronize(s_));
  busy_ = false;
}

}  // namespace gh
