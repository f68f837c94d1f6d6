// Slots of the small V-stack units of the MFMA product (matvec_mfma.hip), host only.
#pragma once
#include <cstddef>

namespace arh {

// Small units per workgroup of `waves` wavefronts, one each: a wavefront per SIMD where there are four, the other
// wavefronts leave at once. Units differ in length, and eight to a workgroup of eight kept its registers until the
// longest was done: FP32 37 rhs 62.5 -> 61 us (58 -> 53.5 us at 1000 Hz, transposed 65 -> 61), FP64 one rhs 48 -> 42
// us; 2, 3, 5 and 6 units are slower than 4.
constexpr std::size_t lr_small(int waves) { return waves < 4 ? waves : 4; }
// Slot u (wavefront u % waves of workgroup u / waves) of the n-th small unit, and the slots of n of them in whole
// workgroups.
constexpr std::size_t lr_slot(std::size_t n, int waves) { return n / lr_small(waves) * waves + n % lr_small(waves); }
constexpr std::size_t lr_slots(std::size_t n, int waves) { return (n + lr_small(waves) - 1) / lr_small(waves) * waves; }

}  // namespace arh
