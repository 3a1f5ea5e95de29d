// The stream of units (query block, delta) that a K-side workgroup walks, with cursors ahead of the unit in work.
#pragma once

namespace sa2 {

constexpr int NEVER = 0x7fffffff;          // the last delta of a block behind the stream: a cursor there stays

// n, or the units from `at` to `stop`, both included, where these are fewer (NEVER - at + 1 would not be an int)
constexpr int units_left(int n, int at, int stop) { return stop - at < n - 1 ? stop - at + 1 : n; }

}  // namespace sa2
