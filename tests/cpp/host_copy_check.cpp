// The host-buffer copies (kf_host_copy.hpp) where threads or memory for them
// run out, and where a chunk's copy fails: the call returns (no exception
// leaves it, none ends the process), with every byte in place or the copy's error.
#include <pthread.h>

#include <dlfcn.h>

#include <cerrno>
#include <cstdint>
#include <cstdio>
#include <new>
#include <vector>

#include "../../acts_amd/csrc/kf_host_copy.hpp"

namespace {
std::atomic<int> failThread{-1};  // this many threads start, no more
std::atomic<int> failNew{-1};     // this many allocations succeed, no more
}  // namespace

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
  if (failThread == 0) return EAGAIN;
  if (failThread > 0) --failThread;
  using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
  return real(t, a, f, x);
}
void* operator new(std::size_t n) {
  if (failNew == 0) throw std::bad_alloc();
  if (failNew > 0) --failNew;
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main() {
  using namespace kf;
  // three arrays, their places 256 bytes apart, over several chunks
  const size_t sizes[] = {size_t{5} << 20, 12345, (size_t{11} << 20) + 7};
  std::vector<char> host[3], back[3];
  CopyPiece in[3], out[3];
  size_t total = 0;
  for (int i = 0; i < 3; ++i) {
    host[i].resize(sizes[i]);
    back[i].resize(sizes[i]);
    for (size_t k = 0; k < sizes[i]; ++k) host[i][k] = static_cast<char>(k * 7 + i);
    in[i] = {host[i].data(), total, sizes[i]};
    out[i] = {back[i].data(), total, sizes[i]};
    total += (sizes[i] + 255) / 256 * 256;
  }
  std::vector<char> dev(total);
  HostCopy copy;
  if (!copy.reserve(total)) return 2;
  int failures = 0;
  auto roundTrip = [&](const char* what, int limit, auto arm) {
    for (int i = 0; i < 3; ++i) std::fill(back[i].begin(), back[i].end(), 0);
    std::fill(dev.begin(), dev.end(), 0);
    arm();
    const hipError_t up = copy.upload(in, 3, dev.data(), total, 0, nullptr);
    arm();
    const hipError_t down = copy.download(out, 3, dev.data(), total, 0, nullptr);
    failThread = failNew = -1;
    bool ok = up == hipSuccess && down == hipSuccess;
    for (int i = 0; i < 3; ++i) ok = ok && back[i] == host[i];
    if (!ok) {
      ++failures;
      std::printf("FAILED %s %d\n", what, limit);
    }
  };
  roundTrip("plain", 0, [] {});
  for (int k = 0; k < 8; ++k) roundTrip("threads", k, [&] { failThread = k; });
  for (int k = 0; k < 8; ++k) roundTrip("memory", k, [&] { failNew = k; });
  for (int k = 0; k < 9; ++k) {
    hipStubFailCopy = k;
    if (copy.upload(in, 3, dev.data(), total, 0, nullptr) == hipSuccess && hipStubFailCopy < 0) {
      ++failures;
      std::printf("FAILED copy error %d not returned\n", k);
    }
    hipStubFailCopy = -1;
    roundTrip("after a copy error", k, [] {});
  }
  copy.release();
  if (failures == 0) std::printf("ok\n");
  return failures ? 1 : 0;
}
