// Unit test of the policy for scratch that a call can do without (final184_amd/csrc/scratch.hpp).
#include <cstdio>
#include <cstdlib>
#include <set>
#include <string>

#include "../../final184_amd/csrc/scratch.hpp"

#define CHECK(c)                                               \
  do {                                                         \
    if (!(c)) {                                                \
      std::printf("CHECK failed line %d: %s\n", __LINE__, #c); \
      std::exit(1);                                            \
    }                                                          \
  } while (0)

struct Device {
  size_t room;  // largest block it gives
  std::set<void*> held;
  std::string log;
  bool drains = true;

  bool reserve(vgi::OptionalScratch& s, size_t need) {
    log.clear();
    return s.reserve(
        need,
        [&](size_t n) -> void* {
          log += 'a';
          if (n > room) return nullptr;
          void* p = std::malloc(1);
          held.insert(p);
          return p;
        },
        [&] { log += 'd'; return drains; },
        [&](void* p) { log += 'r'; CHECK(held.erase(p) == 1); std::free(p); });
  }
};

int main() {
  vgi::OptionalScratch s(1000);
  Device d{600, {}, {}};
  CHECK(d.reserve(s, 100) && d.log == "a" && s.bytes() == 100 && d.held.count(s.data()));
  CHECK(d.reserve(s, 100) && d.reserve(s, 40) && d.log.empty());
  CHECK(d.reserve(s, 101) && d.log == "adr" && s.bytes() == 101 && d.held.size() == 1 && d.held.count(s.data()));
  void* old = s.data();
  // above the limit: nothing is tried, and the block stays
  CHECK(!d.reserve(s, 1001) && d.log.empty() && s.data() == old);
  // not to be had: tried once, nothing drained or freed, the block still serves smaller needs
  CHECK(!d.reserve(s, 700) && d.log == "a" && s.data() == old && s.bytes() == 101);
  CHECK(!d.reserve(s, 700) && d.log.empty());
  CHECK(!d.reserve(s, 900) && d.log.empty());
  CHECK(d.reserve(s, 101) && d.log.empty());
  // a smaller size than the refused one is still tried
  CHECK(d.reserve(s, 500) && d.log == "adr" && s.bytes() == 500 && d.held.size() == 1);
  // the queued work could not be waited for: the old block is kept
  d.drains = false;
  old = s.data();
  CHECK(!d.reserve(s, 550) && d.log == "adr" && s.data() == old && s.bytes() == 500 && d.held.size() == 1);
  std::free(s.data());
  std::printf("SCRATCH OK\n");
  return 0;
}
