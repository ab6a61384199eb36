/*
 * bdem_stage.hpp - the pinned staging buffer between the caller's memory and
 * the device (internal).  Two halves: while one is on its way, the other is
 * copied from or to the caller's arrays.  At most 4 MiB a half whatever the
 * state's size; allocated on first use, given back with its owner.
 */
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

namespace bdem {

/* Large copies are split over a few threads: the caller's fresh pages are
 * faulted in while they are written, which bounds one thread. */
inline void copy_bytes(char* dst, const char* src, size_t len) {
  constexpr size_t SPLIT = 512 * 1024;
  const int parts = (int)std::min<size_t>(4, len / SPLIT);
  if (parts < 2) {
    std::memcpy(dst, src, len);
    return;
  }
  const size_t each = (len / parts + 4095) & ~size_t(4095);
  std::thread th[3];
  int started = 0;
  size_t at = each;   /* [0, each) is this thread's */
  try {
    for (; started < parts - 1 && at < len; ++started, at += each) {
      const size_t o = at, l = std::min(each, len - at);
      th[started] = std::thread([=] { std::memcpy(dst + o, src + o, l); });
    }
  } catch (const std::system_error&) {   /* no thread to be had: the rest is copied here */
  }
  std::memcpy(dst, src, std::min(each, len));
  if (at < len) std::memcpy(dst + at, src + at, len - at);
  for (int k = 0; k < started; ++k) th[k].join();
}

struct HostStage {
  static constexpr size_t HALF_MAX = size_t(4) << 20;
  /* two host arrays that lie one after the other on the device; null: not wanted */
  struct Region {
    char* dev;
    void* h0; size_t n0;
    void* h1; size_t n1;
  };

  HostStage() = default;
  HostStage(const HostStage&) = delete;
  HostStage& operator=(const HostStage&) = delete;
  ~HostStage() { release(); }

  void release() {
    for (hipEvent_t& e : ev) {
      if (e) (void)hipEventDestroy(e);
      e = nullptr;
    }
    if (buf) (void)hipHostFree(buf);
    buf = nullptr;
    half_len = 0;
  }

  hipError_t to_host(const std::vector<Region>& regions, hipStream_t s) {
    hipError_t e = init(regions, s);
    if (e != hipSuccess) return e;
    const std::vector<Piece> p = pieces(regions);
    for (size_t k = 0; k <= p.size(); ++k) {
      if (k < p.size()) {
        e = hipMemcpyAsync(half(k), p[k].r->dev + p[k].off, p[k].len, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipEventRecord(ev[k & 1], s);
        if (e != hipSuccess) break;
      }
      if (k > 0) {
        e = hipEventSynchronize(ev[(k - 1) & 1]);
        if (e != hipSuccess) break;
        exchange(p[k - 1], half(k - 1), true);
      }
    }
    const hipError_t f = hipStreamSynchronize(s);   /* nothing is in flight when an error is returned either */
    return e != hipSuccess ? e : f;
  }

  /* The copies are queued on s; the caller synchronises s before it returns. */
  hipError_t to_device(const std::vector<Region>& regions, hipStream_t s) {
    hipError_t e = init(regions, s);
    if (e != hipSuccess) return e;
    const std::vector<Piece> p = pieces(regions);
    for (size_t k = 0; k < p.size(); ++k) {
      if (k >= 2 && (e = hipEventSynchronize(ev[k & 1])) != hipSuccess) return e;
      exchange(p[k], half(k), false);
      if ((e = hipMemcpyAsync(p[k].r->dev + p[k].off, half(k), p[k].len, hipMemcpyHostToDevice, s)) != hipSuccess)
        return e;
      if ((e = hipEventRecord(ev[k & 1], s)) != hipSuccess) return e;
    }
    return hipSuccess;
  }

 private:
  struct Piece { const Region* r; size_t off, len; };
  char* buf = nullptr;
  size_t half_len = 0;
  hipEvent_t ev[2] = {nullptr, nullptr};

  char* half(size_t k) const { return buf + (k & 1) * half_len; }
  hipError_t init(const std::vector<Region>& regions, hipStream_t s) {
    size_t want = 4096;
    for (const Region& r : regions) want = std::max(want, (r.n0 + r.n1 + 4095) & ~size_t(4095));
    want = std::min(want, HALF_MAX);
    if (half_len < want) {
      if (buf) {
        const hipError_t e = hipStreamSynchronize(s);
        if (e != hipSuccess) return e;
        (void)hipHostFree(buf);
        buf = nullptr;
        half_len = 0;
      }
      const hipError_t e = hipHostMalloc((void**)&buf, 2 * want, hipHostMallocDefault);
      if (e != hipSuccess) {
        buf = nullptr;
        return e;
      }
      half_len = want;
    }
    for (hipEvent_t& x : ev)
      if (!x) {
        const hipError_t e = hipEventCreateWithFlags(&x, hipEventDisableTiming);
        if (e != hipSuccess) {
          x = nullptr;
          return e;
        }
      }
    return hipSuccess;
  }
  std::vector<Piece> pieces(const std::vector<Region>& regions) const {
    std::vector<Piece> p;
    for (const Region& r : regions) {
      size_t o = r.h0 ? 0 : r.n0;
      const size_t end = r.h1 ? r.n0 + r.n1 : (r.h0 ? r.n0 : o);
      for (; o < end; o += half_len) p.push_back(Piece{&r, o, std::min(half_len, end - o)});
    }
    return p;
  }
  /* a piece between its half of the stage and the caller's arrays */
  static void exchange(const Piece& p, char* stage, bool out) {
    auto part = [&](void* h, size_t base, size_t n) {
      if (!h || p.off >= base + n || p.off + p.len <= base) return;
      const size_t a = std::max(p.off, base), b = std::min(p.off + p.len, base + n);
      char* host = static_cast<char*>(h) + (a - base);
      char* st = stage + (a - p.off);
      if (out) copy_bytes(host, st, b - a);
      else copy_bytes(st, host, b - a);
    };
    part(p.r->h0, 0, p.r->n0);
    part(p.r->h1, p.r->n0, p.r->n1);
  }
};

}  // namespace bdem
