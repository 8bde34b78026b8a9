// How many elements of a row a small pull moves together.  Host code of its own, so that it can be tested without a device.
#ifndef TN_ROW_WIDTH_H_
#define TN_ROW_WIDTH_H_

#include <cstdint>

namespace tn {

// The widest of 4, 2 and 1 that divides the rows' length and their distance in the table.
inline int row_width(int wdim, int wstride) { return (wdim | wstride) % 4 == 0 ? 4 : (wdim | wstride) % 2 == 0 ? 2 : 1; }

// ... and suits a variable that stands at `at`.  One element is moved wherever it stands: a caller of the C ABI may hand out a
// float that is not on a boundary of its own.
inline int row_width_at(int width, const void* at) {
    while (width > 1 && reinterpret_cast<uintptr_t>(at) % (width * sizeof(float)) != 0) width /= 2;
    return width;
}

}  // namespace tn

#endif  // TN_ROW_WIDTH_H_
