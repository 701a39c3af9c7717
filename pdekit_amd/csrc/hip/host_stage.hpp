// Copies of results from the device to the caller's memory.
//
// Api: the runtime calls (Hip in rd_method.hip), so that the order of the calls
// can be run without a device.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace pdrd {

// Handed to the runtime directly, a copy to pageable memory is pinned or staged
// page range by page range: 64 KB in 46 us, 512 KB in 248 us, 3.2 MB in 213 us, and
// 29 MB into memory not touched before in 7.6 ms, most of it page faults of the one
// copying thread. Here the data go through a buffer of pinned pieces in groups of
// up to kPieces, copied out while the next pieces of the group arrive, by up to
// kThreads threads where there are several pieces: 18, 36, 130 us and 2.5 ms.
// The buffer (16 MiB) belongs to the process; it is freed with the last method, and
// used by one copy at a time: another thread's copy meanwhile (or one of another
// device) goes to the runtime directly. It is made at the first copy of several
// pieces, or at the second one: making and freeing it takes 45 us (20 of them for the
// events, made with the first copy of several pieces), which a program that reads one
// small field of each of many short-lived methods would pay every time. So does a copy
// to memory that the device reaches itself (pinned, managed or its own): 1 MB 28
// against 70 us through the pieces, 17 MB 304 against 584 us.
template <class Api>
class HostStage
{
public:
  using Error = typename Api::Error;
  using Stream = typename Api::Stream;
  static constexpr size_t kPiece = size_t(1) << 20;
  static constexpr int kPieces = 16, kThreads = 4;

  // one method more or less that may copy
  void user(bool on)
  {
    std::lock_guard<std::mutex> lock(mutex_);
    users_ += on ? 1 : -1;
    if (users_ == 0) drop();
  }

  // n bytes at src (on `device`) to dst, after what the stream holds; complete on
  // return.
  Error copy(int device, Stream stream, void *dst, const void *src, size_t n)
  {
    if (n == 0) return Api::ok;
    std::unique_lock<std::mutex> lock(mutex_, std::defer_lock);
    if (!Api::pageable(dst) || !lock.try_lock() || !ready(device, n > kPiece)) {
      if (lock.owns_lock()) lock.unlock();
      if (Error e = Api::copy(dst, src, n, stream)) return e;
      return Api::wait(stream);
    }
    char *out = static_cast<char *>(dst);
    const char *in = static_cast<const char *>(src);
    if (n <= kPiece) {
      if (Error e = Api::copy(buf_, in, n, stream)) return e;
      if (Error e = Api::wait(stream)) return e;
      std::memcpy(out, buf_, n);
      return Api::ok;
    }
    for (size_t o = 0; o < n; o += kPiece * kPieces)
      if (Error e = group(stream, out + o, in + o, std::min(n - o, kPiece * kPieces))) return e;
    return Api::ok;
  }

private:
  Error group(Stream stream, char *out, const char *in, size_t n)
  {
    const int pieces = static_cast<int>((n + kPiece - 1) / kPiece);
    auto size = [&](int i) { return std::min(kPiece, n - i * kPiece); };
    Error e = Api::ok;
    for (int i = 0; i < pieces && e == Api::ok; ++i) {
      e = Api::copy(buf_ + i * kPiece, in + i * kPiece, size(i), stream);
      if (e == Api::ok) e = Api::record(ev_[i], stream);
    }
    if (e != Api::ok) {
      (void)Api::wait(stream);
      return e;
    }
    // each thread takes the next piece
    std::atomic<int> next{0};
    std::atomic<Error> failed{Api::ok};
    auto work = [&]() noexcept {
      for (int i = next++; i < pieces; i = next++) {
        const Error w = Api::wait(ev_[i]);
        if (w != Api::ok)
          failed = w;
        else
          std::memcpy(out + i * kPiece, buf_ + i * kPiece, size(i));
      }
    };
    std::vector<std::thread> threads;
    try {
      threads.reserve(kThreads);
      for (int t = 1; t < std::min(kThreads, pieces); ++t) threads.emplace_back(work);
    } catch (const std::exception &) {
      // (as many as there are)
    }
    work();
    for (std::thread &t : threads) t.join();
    // (the pieces go to the next copy: none of this one may still arrive)
    if (failed != Api::ok) (void)Api::wait(stream);
    return failed;
  }

  // The buffer for a copy of one piece or of several.
  bool ready(int device, bool several)
  {
    if (!buf_) {
      if (!several && !copied_) {
        copied_ = true;
        return false;
      }
      if (Api::alloc(reinterpret_cast<void **>(&buf_), kPiece * kPieces) != Api::ok) {
        buf_ = nullptr;
        Api::clear_error();
        return false;
      }
      device_ = device;
    }
    if (device_ != device) return false;
    if (!several || ev_[kPieces - 1]) return true;
    bool ok = true;
    for (auto &e : ev_) ok = ok && Api::create(&e) == Api::ok;
    if (!ok) {
      Api::clear_error();
      drop();
    }
    return ok;
  }

  void drop()
  {
    if (buf_) Api::free(buf_);
    buf_ = nullptr;
    for (auto &e : ev_) {
      if (e) Api::destroy(e);
      e = {};
    }
    device_ = -1;
    copied_ = false;
  }

  std::mutex mutex_;
  int users_ = 0;
  int device_ = -1;
  bool copied_ = false;  // a copy has been seen that the buffer was not made for
  char *buf_ = nullptr;
  typename Api::Event ev_[kPieces] = {};
};

}  // namespace pdrd
