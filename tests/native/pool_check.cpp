// Checks of the device memory pool (csrc/pm_pool.h) against a stand-in runtime that counts what it holds.
//   pool_check CASE      exits 0 when the case holds
#include <cstdio>
#include <cstring>
#include <map>
#include <thread>
#include <vector>

#include "pm_pool.h"

namespace {

struct FakeRuntime {
  using Error = int;
  static constexpr Error ok = 0, out_of_memory = 2, invalid = 1;
  struct Live {
    size_t bytes;
    int device;
  };
  static thread_local int device;
  static thread_local std::vector<int> waited;  // devices synchronised by this thread
  static std::mutex mu;
  static std::map<char*, Live> live;
  static size_t capacity, held;
  static char* next;

  // addresses only: nothing is ever stored there
  static Error malloc(void** ptr, size_t bytes) {
    std::lock_guard<std::mutex> lk(mu);
    if (bytes > capacity - held) return out_of_memory;
    *ptr = next;
    live[next] = {bytes, device};
    held += bytes;
    next += (bytes / 4096 + 2) * 4096;
    return ok;
  }
  static Error free(void* ptr) {
    std::lock_guard<std::mutex> lk(mu);
    auto it = live.find((char*)ptr);
    if (it == live.end()) return invalid;
    held -= it->second.bytes;
    live.erase(it);
    return ok;
  }
  static Error range(void** base, size_t* bytes, void* ptr) {
    std::lock_guard<std::mutex> lk(mu);
    auto it = live.upper_bound((char*)ptr);
    if (it == live.begin()) return invalid;
    --it;
    if ((char*)ptr >= it->first + it->second.bytes) return invalid;
    *base = it->first;
    *bytes = it->second.bytes;
    return ok;
  }
  static Error device_of(int* d, void* ptr) {
    std::lock_guard<std::mutex> lk(mu);
    auto it = live.find((char*)ptr);
    if (it == live.end()) return invalid;
    *d = it->second.device;
    return ok;
  }
  static int current_device() { return device; }
  static Error set_device(int d) {
    device = d;
    return ok;
  }
  static Error synchronize() {
    waited.push_back(device);
    return ok;
  }
  static void clear_error() {}
};
thread_local int FakeRuntime::device = 0;
thread_local std::vector<int> FakeRuntime::waited;
std::mutex FakeRuntime::mu;
std::map<char*, FakeRuntime::Live> FakeRuntime::live;
size_t FakeRuntime::capacity = (size_t)64 << 30, FakeRuntime::held = 0;
char* FakeRuntime::next = (char*)0x100000000;

using Pool = pm::DevicePool<FakeRuntime>;
constexpr size_t MiB = (size_t)1 << 20, GiB = (size_t)1 << 30;

#define CHECK(cond)                                                   \
  do {                                                                \
    if (!(cond)) {                                                    \
      std::printf("FAILED %s:%d: %s\n", __FILE__, __LINE__, #cond);   \
      return 1;                                                       \
    }                                                                 \
  } while (0)

void* get(Pool& p, size_t bytes) {
  void* q = nullptr;
  return p.alloc(&q, bytes) == FakeRuntime::ok ? q : nullptr;
}

// a size that cannot be rounded up to whole grains fails; it is not served by a small block
int sizes() {
  Pool p;
  for (size_t bytes : {(size_t)-1, (size_t)-2, (size_t)0 - (pm::kPoolGrain - 1), (size_t)0 - pm::kPoolGrain,
                       (size_t)0 - pm::kPoolGrain - 1, (size_t)1 << 63, 65 * GiB}) {
    void* q = nullptr;
    CHECK(p.alloc(&q, bytes) != FakeRuntime::ok);
    CHECK(q == nullptr && FakeRuntime::held == 0);
  }
  for (size_t bytes : {(size_t)0, (size_t)1, pm::kPoolGrain - 1, pm::kPoolGrain, pm::kPoolGrain + 1, 3 * MiB + 5,
                       pm::kPoolBytes - 1, pm::kPoolBytes, pm::kPoolBytes + 1, 6 * GiB}) {
    void *q = get(p, bytes), *base = nullptr;
    size_t room = 0;
    CHECK(q && FakeRuntime::range(&base, &room, q) == FakeRuntime::ok && base == q && room >= bytes);
    CHECK(p.free(q) == FakeRuntime::ok);
    CHECK(FakeRuntime::held <= pm::kPoolBytes);  // the bound on kept blocks
  }
  p.give_back();
  CHECK(FakeRuntime::held == 0);
  return 0;
}

// an allocation that does not fit next to the kept blocks gets their memory
int pressure() {
  Pool p;
  FakeRuntime::capacity = 4 * GiB;
  void *a = get(p, 1 * GiB), *b = get(p, 2 * GiB);
  CHECK(a && b && p.free(a) == 0 && p.free(b) == 0);
  CHECK(FakeRuntime::held == 3 * GiB);
  void* c = get(p, 3 * GiB + MiB);
  CHECK(c && p.free(c) == 0);
  p.give_back();
  CHECK(FakeRuntime::held == 0);
  return 0;
}

// a block waits for its own device, is handed out on that device alone, and the thread's current device
// stays what it was
int devices() {
  Pool p;
  void* a = get(p, MiB);  // on device 0
  void *other = nullptr, *wrong = nullptr;
  int at = -1, rc = 1;
  std::vector<int> waited;
  std::thread([&] {  // a thread whose current device is another frees it
    FakeRuntime::device = 1;
    rc = p.free(a);
    waited = FakeRuntime::waited;
    at = FakeRuntime::device;
    wrong = get(p, MiB);
    other = get(p, MiB);
    (void)p.free(other);
  }).join();
  CHECK(rc == FakeRuntime::ok && at == 1);
  CHECK(waited == std::vector<int>{0});
  CHECK(wrong != a && other != a);
  CHECK(FakeRuntime::live[(char*)wrong].device == 1);
  CHECK(get(p, MiB) == a);                        // back on its own device, past the other's newer block
  CHECK(p.free(a) == 0 && p.free(wrong) == 0);
  p.give_back();                                  // both devices' blocks
  CHECK(FakeRuntime::held == 0);
  return 0;
}

// the scratch buffer grows to the largest request, is kept between calls up to its bound, and goes back
// under pressure and on request unless a call uses it
int scratch() {
  Pool p;
  FakeRuntime::capacity = 4 * GiB;
  void* a = p.scratch(300 * MiB);
  CHECK(a && FakeRuntime::held == 300 * MiB);
  p.give_back();
  CHECK(FakeRuntime::held == 300 * MiB);           // in use
  void* big = nullptr;
  CHECK(p.plain_alloc(&big, 4 * GiB) != FakeRuntime::ok && FakeRuntime::held == 300 * MiB);
  p.scratch_done();
  CHECK(p.scratch(200 * MiB) == a);                // kept, large enough
  p.scratch_done();
  CHECK(p.plain_alloc(&big, 4 * GiB) == FakeRuntime::ok && FakeRuntime::held == 4 * GiB);  // idle: given back
  CHECK(p.scratch(MiB) == nullptr);                // no memory: the call does without
  p.scratch_done();
  CHECK(FakeRuntime::free(big) == FakeRuntime::ok);
  CHECK(p.scratch(2 * GiB) && FakeRuntime::held == 2 * GiB);
  p.scratch_done();
  CHECK(FakeRuntime::held == 0);                   // above the bound: not kept
  CHECK(p.scratch(500 * MiB) && p.scratch(600 * MiB) && FakeRuntime::held == 600 * MiB);
  p.scratch_done();
  p.give_back();
  CHECK(FakeRuntime::held == 0);
  return 0;
}

}  // namespace

int main(int argc, char** argv) {
  const char* name = argc > 1 ? argv[1] : "";
  int rc = 2;
  if (!std::strcmp(name, "sizes")) rc = sizes();
  if (!std::strcmp(name, "pressure")) rc = pressure();
  if (!std::strcmp(name, "devices")) rc = devices();
  if (!std::strcmp(name, "scratch")) rc = scratch();
  if (rc == 0) std::printf("%s: ok\n", name);
  return rc;
}
