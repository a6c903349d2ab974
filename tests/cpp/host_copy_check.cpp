// The host-side copy helpers against plain memcpy: random job lists (many small pieces, a few
// large ones, empty ones) through host_copy, blocks in units through host_copy_units as the staging
// paths move them, with errors, exceptions and a shortage of threads on the way; every thread count, with the
// bytes around every destination checked for overruns.  Built with AddressSanitizer and with ThreadSanitizer by
// tests/test_host_cpp.py; needs no GPU.  Prints "host_copy_check ok <cases>" and "host_copy_units ok <cases>".
#include <pthread.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <random>
#include <stdexcept>
#include <thread>
#include <vector>

#include "axr_internal.h"

namespace {

// A block of `span` bytes copied in units.  `fail_at`: done() of that unit returns an error, or throws.
struct CopyUnits : axr::HostUnits {
  const uint8_t* src;
  uint8_t* dst;
  size_t told = 0, fail_at = SIZE_MAX;
  bool throws = false, in_order = true;
  std::unique_ptr<std::atomic<uint8_t>[]> seen;
  CopyUnits(size_t bytes, size_t unit_bytes, size_t threads, const uint8_t* from, uint8_t* to) : src(from), dst(to) {
    span = bytes;
    unit = unit_bytes;
    helpers = threads - 1;
    seen.reset(new std::atomic<uint8_t>[bytes / unit_bytes + 2]());
  }
  bool ready(size_t, bool) override { return true; }
  void copy(size_t lo, size_t hi) override {
    seen[lo / unit].fetch_add(1);
    std::memcpy(dst + lo, src + lo, hi - lo);
  }
  int done(size_t u) override {
    in_order = in_order && u == told && std::memcmp(dst + u * unit, src + u * unit, std::min(unit, span - u * unit)) == 0;
    ++told;
    if (u != fail_at) return AXR_OK;
    if (throws) throw std::runtime_error("done");
    return AXR_ERR_HIP;
  }
};

constexpr int kThrows = 1001, kNoFlags = 1002;

// A "device" that fills a block from the front and raises its flags, slower than they are looked at.
struct ArrivingUnits : axr::FlaggedUnits {
  std::vector<uint8_t> staged, out;
  std::vector<uint32_t> up;
  const std::vector<uint8_t>& src;
  size_t stall_at;        // no flag from this one on before the host waits
  int fails;              // arrive(): 0, an error, or kThrows, or kNoFlags: returns without the flags
  bool waited = false;
  std::atomic<bool> asked{false};
  std::thread device;
  ArrivingUnits(const std::vector<uint8_t>& from, size_t unit_bytes, size_t piece_bytes, size_t threads, size_t stall, int how)
      : staged(from.size()), out(from.size(), 0), src(from), stall_at(stall), fails(how) {
    span = from.size();
    unit = unit_bytes;
    helpers = threads - 1;
    piece = piece_bytes;
    looks = 50;
    up.assign((span + piece - 1) / piece, 0);
    flags = up.data();
    device = std::thread([this] {
      for (size_t i = 0; i < up.size(); ++i) {
        while (i >= stall_at && !asked.load()) std::this_thread::yield();
        if (fails && i >= stall_at) return;
        const size_t lo = i * piece, hi = std::min(lo + piece, span);
        std::memcpy(staged.data() + lo, src.data() + lo, hi - lo);
        __atomic_store_n(&up[i], 1u, __ATOMIC_RELEASE);
      }
    });
  }
  ~ArrivingUnits() override {
    asked = true;
    if (device.joinable()) device.join();
  }
  int arrive() override {
    waited = true;
    asked = true;
    if (device.joinable()) device.join();
    if (fails == kThrows) throw std::runtime_error("arrive");
    return fails == kNoFlags ? AXR_OK : fails;
  }
  void copy(size_t lo, size_t hi) override { std::memcpy(out.data() + lo, staged.data() + lo, hi - lo); }
  int done(size_t) override { return AXR_OK; }
};

int bad(const char* what, long at) {
  std::fprintf(stderr, "host_copy_units: %s (case %ld)\n", what, at);
  return 1;
}

// A block goes to the payload in at most four transfers, whatever its length.
int check_pieces() {
  std::mt19937_64 rng(13);
  for (int i = 0; i < 20000; ++i) {
    const size_t around = (size_t{1} << 18) * (1 + i % 32);
    const size_t span = i < 200 ? around + i / 32 * 5 - 15 : 1 + rng() % (8u << 20);
    size_t sent = 0, transfers = 0;
    for (size_t at = 0; at < span;) {
      at = std::min(at + axr::kStageUnit, span);
      if (at < span && at - sent < axr::stage_piece(span, sent)) continue;
      sent = at;
      ++transfers;
    }
    if (transfers > 4 || (span <= axr::kStageSend && transfers != 1)) return bad("transfers of a block", static_cast<long>(span));
  }
  return 0;
}

int check_units() {
  std::mt19937_64 rng(12);
  auto pick = [&](uint64_t lo, uint64_t hi) { return lo + rng() % (hi - lo + 1); };
  long cases = 0;
  for (int round = 0; round < 30; ++round) {
    const size_t unit = pick(1, 3) == 1 ? pick(1, 100) : pick(1000, 70000);
    const size_t span = round == 0 ? 0 : unit * pick(0, 40) + pick(round == 1 ? 0 : 1, unit);
    std::vector<uint8_t> src(span + 1);
    for (uint8_t& b : src) b = static_cast<uint8_t>(rng());
    const size_t n = (span + unit - 1) / unit;
    for (size_t threads : {1, 2, 4, 16}) {
      for (int how = 0; how < 4; ++how, ++cases) {   // to the end, an error, an exception, no thread to be had
        std::vector<uint8_t> dst(span + 64, 0xEE);
        CopyUnits units(span, unit, threads, src.data(), dst.data() + 32);
        if ((how == 1 || how == 2) && n) units.fail_at = pick(0, n - 1);
        units.throws = how == 2;
        pthread_attr_t usual, huge;
        if (how == 3) {   // stacks that no address space holds
          pthread_getattr_default_np(&usual);
          pthread_attr_init(&huge);
          pthread_attr_setstacksize(&huge, size_t{1} << 47);
          if (pthread_setattr_default_np(&huge) != 0) return bad("stack size", cases);
        }
        int rc = AXR_OK;
        bool threw = false;
        try {
          rc = axr::host_copy_units(units);
        } catch (const std::runtime_error&) {
          threw = true;
        }
        if (how == 3) pthread_setattr_default_np(&usual);
        const bool fails = units.fail_at != SIZE_MAX;
        if (threw != (fails && units.throws) || (rc != AXR_OK) != (fails && !units.throws)) return bad("outcome", cases);
        if (!units.in_order || units.told != (fails ? units.fail_at + 1 : n)) return bad("done out of turn", cases);
        for (size_t u = 0; u < n; ++u)
          if (units.seen[u] > 1 || (!fails && units.seen[u] != 1)) return bad("units", cases);
        if (!fails && std::memcmp(dst.data() + 32, src.data(), span) != 0) return bad("bytes", cases);
        for (size_t i = 0; i < 32; ++i)
          if (dst[i] != 0xEE || dst[span + 32 + i] != 0xEE) return bad("overrun", cases);
      }
    }
  }
  for (int round = 0; round < 30; ++round) {
    const size_t piece = pick(1, 2) == 1 ? 16384 : pick(10, 3000), unit = piece * pick(1, 5);
    std::vector<uint8_t> src(unit * pick(0, 20) + pick(1, unit));
    for (uint8_t& b : src) b = static_cast<uint8_t>(rng());
    const size_t pieces = (src.size() + piece - 1) / piece;
    for (size_t threads : {1, 2, 4, 16})
      for (int fails : {0, static_cast<int>(AXR_ERR_HIP), kThrows, kNoFlags}) {
        const size_t stall = fails || round % 2 ? pick(0, pieces - 1) : SIZE_MAX;
        ArrivingUnits units(src, unit, piece, threads, stall, fails);
        int rc = AXR_OK;
        bool threw = false;
        try {
          rc = axr::host_copy_units(units);
        } catch (const std::runtime_error&) {
          threw = true;
        }
        if (rc != AXR_OK || threw != (fails == kThrows)) return bad("flagged outcome", cases);
        if ((units.status != AXR_OK) != (fails != 0 && fails != kThrows)) return bad("flagged status", cases);
        if (stall != SIZE_MAX && !units.waited) return bad("not waited for", cases);
        if (!fails && units.out != src) return bad("flagged bytes", cases);
        ++cases;
      }
  }
  std::printf("host_copy_units ok %ld\n", cases);
  return 0;
}

}  // namespace

int main() {
  std::mt19937_64 rng(11);
  auto pick = [&](uint64_t lo, uint64_t hi) { return lo + rng() % (hi - lo + 1); };
  long cases = 0;
  for (int round = 0; round < 25; ++round) {
    const size_t njobs = pick(0, 40);
    std::vector<size_t> sizes(njobs);
    size_t total = 0;
    for (size_t& n : sizes) {
      const uint64_t kind = pick(0, 9);
      n = kind == 0 ? 0 : (kind < 7 ? pick(1, 70000) : pick(1u << 20, 5u << 20));
      total += n;
    }
    std::vector<uint8_t> src(total + 1), want(total + 64 * (njobs + 1), 0xEE), got;
    for (size_t i = 0; i < total; ++i) src[i] = static_cast<uint8_t>(rng());
    // destinations: 32 guard bytes between jobs
    std::vector<axr::HostCopyJob> jobs(njobs);
    got = want;
    size_t s_at = 0, d_at = 32;
    for (size_t j = 0; j < njobs; ++j) {
      std::memcpy(want.data() + d_at, src.data() + s_at, sizes[j]);
      jobs[j] = {got.data() + d_at, src.data() + s_at, sizes[j]};
      s_at += sizes[j];
      d_at += sizes[j] + 32;
    }
    for (int64_t threads : {1, 2, 3, 4, 7, 16}) {
      if (axr_tune_set("host_threads", threads) != AXR_OK) return 1;
      std::vector<uint8_t> out = got;   // fresh guard pattern every time
      std::vector<axr::HostCopyJob> mine = jobs;
      for (axr::HostCopyJob& job : mine)
        job.dst = out.data() + (static_cast<uint8_t*>(job.dst) - got.data());
      axr::host_copy(mine.data(), mine.size());
      if (out != want) {
        std::fprintf(stderr, "host_copy_check: mismatch in round %d with %lld threads\n", round,
                     static_cast<long long>(threads));
        return 1;
      }
      ++cases;
    }
  }
  std::printf("host_copy_check ok %ld\n", cases);
  return check_pieces() + check_units();
}
