// row_extent.h — how many bytes of a row of logits its buffer descriptor serves (sampler.hip).
// Plain C++: the host tests compile it.
#pragma once

#include <stdint.h>

namespace dsv41 {

// Loads of one element are range-checked by the element, so the row ends where it ends: one byte
// more could lie on the next page when a bf16 row begins between two dwords.  Vector loads, whose
// rows begin on a 16-byte boundary, are checked dword by dword: the dword that holds an odd bf16
// row's last id is served whole, with one element past the row that the kernels mask by V.
constexpr uint32_t row_extent(int V, int esize, bool vec) {
  return vec ? ((uint32_t)V * (uint32_t)esize + 3u) & ~3u : (uint32_t)V * (uint32_t)esize;
}

}  // namespace dsv41
