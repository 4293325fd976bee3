// epet_plan.hpp -- decisions on sizes alone (host code without device types).
#pragma once

namespace epet {

// Whether to try again what memory was too short for when `short_at` bytes were
// available (0: not tried): only with an eighth and 64 MB more.  An attempt copies
// row ids, sorts them on the host and waits for the device when it fails (20 ns per
// row and column), which a caller short of memory would pay on every call.
inline bool memory_worth_trying(unsigned long long available, unsigned long long short_at) {
  return short_at == 0 || available > short_at + short_at / 8 + (64ull << 20);
}

// Bytes that bricks of both directions take at least: `parts` halfwords an entry.
inline unsigned long long bricks_at_least(long long nnz, int parts) {
  return 4ull * (unsigned long long)parts * (unsigned long long)nnz;
}

}  // namespace epet
