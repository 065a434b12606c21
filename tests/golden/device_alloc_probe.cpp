// Device allocations of a process, checked: loaded with global symbols before
// the library, its hipMalloc is the one the library calls.  Every allocation
// gets a guard of 256 bytes behind the size asked for, and one allocation can
// be made to fail.
#include <dlfcn.h>

#include <cstddef>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
constexpr size_t kGuard = 256;
constexpr int kOutOfMemory = 2, kToHost = 2, kToDevice = 1;
std::map<void*, size_t> live;
std::string failure;
long count = 0, fail_at = -1;
size_t fail_from = 0;

template <class F>
F real(const char* name) {
  static void* lib = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL);
  return reinterpret_cast<F>(dlsym(lib, name));
}
using Malloc = int (*)(void**, size_t);
using Free = int (*)(void*);
using Copy = int (*)(void*, const void*, size_t, int);
}  // namespace

extern "C" {
int hipMalloc(void** p, size_t bytes) {
  const long k = count++;
  if (k == fail_at || (fail_from && bytes >= fail_from)) {
    // the runtime's own refusal, so that it also leaves its error behind
    return real<Malloc>("hipMalloc")(p, size_t(1) << 60);
  }
  const int e = real<Malloc>("hipMalloc")(p, bytes + kGuard);
  if (e) return e;
  std::vector<unsigned char> g(kGuard, 0xa5);
  real<Copy>("hipMemcpy")(static_cast<char*>(*p) + bytes, g.data(), kGuard, kToDevice);
  live[*p] = bytes;
  return 0;
}

int hipFree(void* p) {
  live.erase(p);
  return real<Free>("hipFree")(p);
}

// allocations asked for so far
long probe_count() { return count; }
long probe_live() { return static_cast<long>(live.size()); }
long probe_bytes() {
  long n = 0;
  for (const auto& a : live) n += static_cast<long>(a.second);
  return n;
}
// the k-th allocation from now fails (-1: none)
void probe_fail(long k) { fail_at = k < 0 ? -1 : count + k; }
// every allocation of at least this many bytes fails (0: none)
void probe_fail_from(size_t bytes) { fail_from = bytes; }

// allocations whose guard was written to
long probe_damaged() {
  long bad = 0;
  std::vector<unsigned char> g(kGuard);
  for (const auto& a : live) {
    real<Copy>("hipMemcpy")(g.data(), static_cast<char*>(a.first) + a.second, kGuard, kToHost);
    for (unsigned char c : g)
      if (c != 0xa5) {
        ++bad;
        break;
      }
  }
  return bad;
}
}
