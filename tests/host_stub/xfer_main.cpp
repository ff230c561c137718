// Host tests of the transfer ring (csrc/mge_xfer.h) on the stand-in runtime;
// argv[1] names the test, the exit status is 0 if it holds.
#include <cstdio>
#include <string>

#include "mge_xfer.h"

using namespace mge;

static bool round_trip(StubStream &st, size_t n, unsigned seed) {
  std::vector<char> dev(n), in(n), out(n, 0);
  for (size_t q = 0; q < n; q++) in[q] = (char)((q * 2654435761u + seed) >> 13);
  hipError_t e = xfer(st.dev, &st, dev.data(), n, true,
                      [&](size_t o, char *t, size_t len) { std::memcpy(t, in.data() + o, len); });
  if (e == hipSuccess && dev != in) {
    std::printf("%zu bytes up: wrong\n", n);
    return false;
  }
  if (e == hipSuccess)
    e = xfer(st.dev, &st, dev.data(), n, false,
             [&](size_t o, const char *t, size_t len) { std::memcpy(out.data() + o, t, len); });
  if (e != hipSuccess || out != in) {
    std::printf("%zu bytes: error %d, %s\n", n, (int)e, out == in ? "right" : "wrong");
    return false;
  }
  return true;
}

// small ones, whole pieces, ragged tails, more pieces than the ring has places
static bool sizes() {
  StubStream st(0);
  bool ok = true;
  for (size_t n : {size_t(1), size_t(1000), kPiece, 2 * kPiece, 2 * kPiece + 8, 7 * kPiece - 24, 8 * kPiece,
                   17 * kPiece + 40, 25 * kPiece})
    ok = round_trip(st, n, 1) && ok;
  return ok;
}

static bool threads() {
  std::atomic<int> bad{0};
  std::vector<std::thread> ts;
  for (int t = 0; t < 4; t++)
    ts.emplace_back([&, t] {
      hipSetDevice(t % 2);
      StubStream st(t % 2);
      if (!round_trip(st, (4 + 6 * t) * kPiece + 8 * t, t) || !round_trip(st, 1000 + t, t)) bad++;
    });
  for (auto &t : ts) t.join();
  return bad == 0;
}

// a thread whose current device is not the case's
static bool device() {
  StubStream st(0);
  hipSetDevice(1);
  const bool ok = round_trip(st, 20 * kPiece + 8, 3) && round_trip(st, 100, 3);
  int d = -1;
  hipGetDevice(&d);
  std::printf("current device %d\n", d);
  return ok && d == 1;
}

// transfers of another case while `n` are stuck in their callers' memory
static bool beside(int n) {
  std::atomic<int> entered{0}, release{0}, done{0}, ok{0};
  std::vector<std::thread> big;
  for (int t = 0; t < n; t++)
    big.emplace_back([&] {
      StubStream st(0);
      std::vector<char> dev(20 * kPiece);
      xfer(0, &st, dev.data(), dev.size(), false, [&](size_t o, const char *, size_t) {
        if (o == 0) entered++;
        while (!release) std::this_thread::yield();
      });
    });
  for (int t = 0; t < 1000 && entered < n; t++) std::this_thread::sleep_for(std::chrono::milliseconds(5));
  std::thread other([&] {
    StubStream st(0);
    ok = round_trip(st, 1000, 5) && round_trip(st, 11 * kPiece + 16, 5);
    done = 1;
  });
  for (int t = 0; t < 2000 && !done; t++) std::this_thread::sleep_for(std::chrono::milliseconds(5));
  const bool in_time = done != 0;
  release = 1;
  for (auto &t : big) t.join();
  other.join();
  std::printf("finished beside %d: %d\n", n, (int)in_time);
  return in_time && ok;
}

// no pinned memory to be had
static bool unpinned() {
  stub_no_pinned = 1;
  StubStream st(0);
  return round_trip(st, 5 * kPiece + 8, 6) && round_trip(st, 10, 6);
}

int main(int argc, char **argv) {
  const std::string t = argc > 1 ? argv[1] : "";
  xfer_user(1);
  const bool ok = t == "sizes" ? sizes() : t == "threads" ? threads() : t == "device" ? device()
                  : t == "beside_one" ? beside(1) : t == "beside_five" ? beside(5) : t == "unpinned" ? unpinned() : false;
  xfer_user(-1);
  return ok ? 0 : 1;
}
