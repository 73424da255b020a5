// prefill_span.h -- how many pages the keys of one prefill workgroup can touch.
// Plain C++, so that the rule can be checked on the host alone.
#pragma once
#include <algorithm>
#include <cstdint>

namespace sandy_hip {

// Keys 0 .. tk - 1 in pages of 1 << log2_page rows; a workgroup's 32 * rw rows are
// neighbouring queries of `group` heads each, every query seeing the `window` keys
// up to its own (window <= 0: all before it).  A window of tk keys or more bounds
// nothing: callers pass values up to INT64_MAX for "no limit", so nothing is added
// to a window before that is known.
inline int64_t prefill_page_span(int64_t tk, int64_t window, int64_t rw, int64_t group, int log2_page) {
    const int64_t all = (tk >> log2_page) + 1;
    if (window <= 0 || window >= tk) return all;
    return std::min(all, ((window + 32 * rw / group + 1) >> log2_page) + 2);
}

} // namespace sandy_hip
