// Values that one workgroup hands to a persistent kernel's others over a grid barrier, as plain
// code (no HIP calls), so that it can be checked on the host without a GPU.
//
// They are stored before the barrier that ends pass R and read by everyone after it.
// The next pass may begin with a phase that the storing workgroup runs alone, and end it
// while others have yet to read: so pass R + 1 stores elsewhere.  Pass R + 2 stores after
// the barrier of pass R + 1, to which every reader of pass R has come by then.
#pragma once

namespace indigo {

template <typename T>
struct ByPass {
  T slot[2];
  constexpr T& of(int pass) { return slot[pass & 1]; }
};

}  // namespace indigo
