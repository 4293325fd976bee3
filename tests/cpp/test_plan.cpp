// Decisions on sizes alone (epet_plan.hpp), compiled without HIP.
#include <cstdio>

#include "../../epetreco_amd/csrc/epet_plan.hpp"

static int fails = 0;
static void check(bool ok, const char* what) {
  std::printf("%s %s\n", ok ? "ok  " : "FAIL", what);
  fails += !ok;
}

int main() {
  using namespace epet;
  const unsigned long long GB = 1ull << 30;
  check(memory_worth_trying(0, 0), "the first attempt is made whatever is known of the memory");
  check(!memory_worth_trying(10 * GB, 10 * GB), "not again with the same memory");
  check(!memory_worth_trying(9 * GB, 10 * GB), "nor with less");
  check(!memory_worth_trying(11 * GB, 10 * GB), "nor with little more");
  check(memory_worth_trying(12 * GB, 10 * GB), "again with clearly more");
  check(!memory_worth_trying(1, 1) && !memory_worth_trying(64ull << 20, 1), "nothing available once");
  check(memory_worth_trying(65ull << 20, 1), "and something later");
  check(bricks_at_least(3000000000ll, 3) == 36000000000ull, "entries beyond 31 bits");
  check(bricks_at_least(0, 1) == 0, "no entries");
  std::printf("%s: %d failure(s)\n", fails ? "FAILED" : "PASSED", fails);
  return fails != 0;
}
