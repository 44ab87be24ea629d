// Runs the host copies of nlm_copy.hip on a CPU, over the runtime in fake_hip/, one scenario
// per run (argv[1]); exits 0 if every check holds.
#include <dlfcn.h>
#include <pthread.h>

#include <cstdio>
#include <vector>

#include "../multimodenonlinearoptics_amd/csrc/nlm_copy.hip"

int set_err(int kind, const std::string& msg) {
  std::printf("error: %s\n", msg.c_str());
  return kind;
}

static std::atomic<int> threadsAllowed{1 << 30}, threadsMade{0};
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
  using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Fn real = (Fn)dlsym(RTLD_NEXT, "pthread_create");
  if (threadsAllowed <= 0) return EAGAIN;
  threadsAllowed--;
  threadsMade++;
  return real(t, a, f, x);
}

static int failures = 0;
#define CHECK(x) \
  do { \
    if (!(x)) std::printf("line %d: %s\n", __LINE__, #x), failures++; \
  } while (0)

// Results of the given sizes, copied in one call; every byte has to arrive.
static void copy(const std::vector<size_t>& sizes, FakeStream* s, unsigned seed) {
  std::vector<std::vector<char>> dev, host;
  std::vector<HostCopy> items;
  for (size_t k = 0; k < sizes.size(); k++) {
    dev.emplace_back(sizes[k]);
    host.emplace_back(sizes[k], (char)0x5a);
    for (size_t i = 0; i < sizes[k]; i++) dev[k][i] = (char)(i * 31 + (i >> 9) + seed + k);
  }
  for (size_t k = 0; k < sizes.size(); k++) items.push_back({host[k].data(), dev[k].data(), sizes[k]});
  items.push_back({nullptr, nullptr, 100});
  CHECK(nlm_to_host(items.data(), (int)items.size(), s) == NLM_OK);
  for (size_t k = 0; k < sizes.size(); k++) CHECK(dev[k] == host[k]);
}

constexpr size_t MB = (size_t)1 << 20;

// A second caller's large copy, in the middle of a first one's
static void second() {
  std::thread([] {
    FakeStream s{0};
    std::vector<char> dev(4 * MB, 3), host(4 * MB, 0);
    fake::watched = host.data();
    const HostCopy c = {host.data(), dev.data(), host.size()};
    CHECK(nlm_to_host(&c, 1, &s) == NLM_OK);
    CHECK(fake::watchedCopies == 1 && dev == host);
  }).join();
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  FakeStream s{0};
  if (what == "sizes") {
    for (unsigned r = 0; r < 3; r++) {
      copy({1, 100, 256 << 10, (256 << 10) + 1, MB}, &s, r);
      copy({3 * MB - 1, 3 * MB, 3 * MB + 7, 17, 9 * MB + 5, 300000, 64}, &s, r);
      copy(std::vector<size_t>(40, 255 << 10), &s, r);  // more than the area holds
    }
    CHECK(threadsMade == 3);
  } else if (what == "helpers") {
    // only one helper can be started at first, later all of them
    threadsAllowed = 1;
    copy({5 * MB}, &s, 0);
    CHECK(threadsMade == 1);
    threadsAllowed = 1 << 30;
    for (unsigned r = 0; r < 20; r++) copy({13 * MB + r}, &s, r);
    CHECK(threadsMade == 3);
  } else if (what == "no area") {
    fake::failHostMalloc = true;
    copy({100, MB, 5 * MB}, &s, 0);
    fake::failHostMalloc = false;
    fake::failEventCreate = true;
    copy({100, MB, 5 * MB}, &s, 1);
    CHECK(fake::areas == 0 && fake::events == 0 && hipGetLastError() == hipSuccess);
    fake::failEventCreate = false;
    copy({100, MB, 5 * MB}, &s, 2);
    CHECK(fake::areas == 1);
  } else if (what == "device") {
    FakeStream other{1};
    for (unsigned r = 0; r < 2; r++) {
      copy({100, 5 * MB}, &other, r);
      CHECK(fake::device == 0);
      copy({100, 5 * MB}, &s, r);
    }
    CHECK(fake::areas == 2);
  } else if (what == "pinned") {
    // two results in pinned memory, one large and one small, between two in ordinary memory
    std::vector<char> dev(5 * MB, 7), pin(6 * MB, 0), a(100, 0), b(4 * MB, 0);
    fake::pinned = pin.data();
    fake::pinnedEnd = pin.data() + pin.size();
    const HostCopy c[] = {{a.data(), dev.data(), 100}, {pin.data(), dev.data(), 5 * MB},
                          {b.data(), dev.data(), 4 * MB}, {pin.data() + 5 * MB, dev.data(), 200}};
    CHECK(nlm_to_host(c, 4, &s) == NLM_OK);
    CHECK(fake::pinnedCopies == 2);
    for (size_t i = 0; i < pin.size(); i++)
      if (pin[i] != (i < 5 * MB + 200 ? 7 : 0)) failures++;
    for (char x : a) failures += x != 7;
    for (char x : b) failures += x != 7;
  } else if (what == "two callers") {
    for (int r = 1; r <= 3; r++) {
      fake::watchedCopies = 0;
      fake::onCopy = second;
      copy({9 * MB}, &s, r);
    }
    CHECK(threadsMade == 3 + 3);  // helpers, and the second callers themselves
  } else if (what == "one cpu") {
    cpu_set_t all, one;
    sched_getaffinity(0, sizeof all, &all);
    CPU_ZERO(&one);
    for (int k = 0; k < CPU_SETSIZE && CPU_COUNT(&one) == 0; k++)
      if (CPU_ISSET(k, &all)) CPU_SET(k, &one);
    sched_setaffinity(0, sizeof one, &one);
    second();
    CHECK(threadsMade == 1);  // the caller itself
  } else {
    std::printf("unknown scenario\n");
    return 2;
  }
  return failures ? 1 : 0;
}
