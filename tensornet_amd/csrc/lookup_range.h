// The lookups of an example, as the forward combiner's workgroup finds them.  Code of its own, so that it can be tested without a
// device.
#ifndef TN_LOOKUP_RANGE_H_
#define TN_LOOKUP_RANGE_H_

#include <cstdint>

namespace tn {

struct LookupRange {
    uint32_t from, to;
};

// Of the lookups [lo, hi) a workgroup has looked at, those of an example: `first` is the position that started it and `behind` the
// one behind its last lookup, each 0 if no lookup was that.  In order a lookup that ends an example has one that starts it; out of
// order the start may have been refused and the end not, and such an example has none: whatever the ids, a range that is not
// empty lies in [lo, hi).
constexpr LookupRange lookup_range(uint32_t first, uint32_t behind, uint32_t lo) {
    return {first, first < lo || behind < first ? first : behind};
}

}  // namespace tn

#endif  // TN_LOOKUP_RANGE_H_
