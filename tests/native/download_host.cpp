// download() on the CPU, over a stand-in for the HIP runtime. Arguments: what
// to check. Exit status 0: as it should be.
#include <cstdio>
#include <cstdlib>
#include <new>
#include <string>
#include <vector>

#include "internal.hpp"

namespace {
thread_local long g_fail_at = 0;  // this thread's allocation that fails (1: the next)
}

void* operator new(size_t n) {
  if (g_fail_at > 0 && --g_fail_at == 0) throw std::bad_alloc();
  void* p = std::malloc(n == 0 ? 1 : n);
  if (p == nullptr) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  std::vector<char> from(size_t(37) << 20), to(from.size());
  for (size_t i = 0; i < from.size(); ++i) from[i] = static_cast<char>(i * 2654435761u >> 13);
  msim::Context ctx;
  msim::download_enter();
  int bad = 0;
  auto expect = [&](bool ok, const char* text) {
    if (!ok) std::printf("%s: %s\n", what.c_str(), text), ++bad;
  };
  auto get = [&] {
    std::fill(to.begin(), to.end(), 0);
    fake_copies = 0;
    msim::download(ctx, to.data(), from.data(), from.size(), "download");
    return to == from;
  };
  if (what == "registered") {
    fake_registered = to.data();
    expect(get() && fake_copies == 1, "a destination the runtime can write goes in one copy");
    fake_registered = nullptr;
    expect(get() && fake_copies == 19, "another goes through the slots");
  } else if (what == "allocations") {
    // Each allocation of the calling thread fails once: the call ends with the
    // bytes or with bad_alloc, and no slot is lost to later calls.
    expect(get(), "the bytes");
    const int slots = fake_slots;
    for (long k = 1; k < 60; ++k) {
      g_fail_at = k;
      try {
        msim::download(ctx, to.data(), from.data(), from.size(), "download");
        if (g_fail_at > 0) break;  // it makes fewer
      } catch (const std::bad_alloc&) {
      }
      g_fail_at = 0;
      expect(get() && fake_copies == 19, "the bytes after a failed allocation");
      expect(fake_slots == slots, "the slots after a failed allocation");
    }
    g_fail_at = 0;
  }
  msim::download_leave();
  expect(fake_slots == 0, "the slots go with the last context");
  return bad;
}
