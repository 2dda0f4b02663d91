// The extent and the scalar offset of a raw buffer load of one group of K. Plain C++: host code can evaluate it too.
#pragma once

namespace sepal::hip {

struct Window {
    unsigned bytes;  // the descriptor's extent
    int scalar;      // the load's scalar offset
};

// Kernels that keep the loads of every step alike load a group past their range through an empty window: zeros and no
// memory access. Its scalar offset is 0 as well: a range check that compares the lane's offset with extent - scalar would
// wrap for an extent of 0 beside a larger scalar offset, and the load would read past the operand's end.
constexpr Window group_window(bool in, unsigned bytes, int scalar) { return in ? Window{bytes, scalar} : Window{0u, 0}; }

} // namespace sepal::hip
