// Which synchronous reads of a caller's address a kernel may do (Ctx::read_column).
#pragma once
#include <cstddef>
#include <cstdint>
#include <unordered_map>

namespace sh {

// The columns that a context has handed out: first address -> bytes.
using LiveColumns = std::unordered_map<void*, size_t>;

// Whether words [first, first + words) of col lie in a live column that begins at col. Any other address
// (inside a column, of another context, a caller's own memory, the host's, stale) is left to the copy
// engine, which can refuse it; a kernel that read it could only fault.
inline bool kernel_may_read(const LiveColumns& live, const uint32_t* col, size_t first, size_t words) {
  const auto it = live.find(const_cast<uint32_t*>(col));
  if (it == live.end()) return false;
  const size_t held = it->second / 4;
  return first <= held && words <= held - first;
}

}  // namespace sh
