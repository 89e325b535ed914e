// Byte offsets of the reads of a product's operands (gemm_f32.hip): plain arithmetic, for the kernel and for checks on a host.
//
// An operand is read through a buffer descriptor of its size: a scalar offset for the step of the contraction and a vector
// offset for a lane's place in the step.  The hardware refuses a vector offset that is not below the size less the scalar
// offset, so the scalar one never exceeds the size: steps that are asked for ahead of time, past the last one, keep the last
// one's and take a vector offset that no operand reaches.
#pragma once
#include <cstdint>

namespace t5a {

constexpr int kGemmStep = 32;            // contraction indices of a staged tile
constexpr int kNoRead = 0x7fffffe0;      // (operands are smaller than 0x7ff00000 bytes; 16 more do not overflow)

// from the first byte to the last of `lines` lines of `width` elements, `ld` apart
constexpr int operand_bytes(int lines, int width, int64_t ld, int size) { return (int)(((lines - 1) * ld + width) * size); }
// between two steps; `ld` where the contraction's indices are lines, else 1
constexpr int step_bytes(int K, int64_t ld, int size) { return K > kGemmStep ? (int)(kGemmStep * ld * size) : 0; }
constexpr int step_offset(int kk, int K, int step) { return (kk < (K - 1) / kGemmStep ? kk : (K - 1) / kGemmStep) * step; }
// of a lane whose index in the step is k
constexpr int lane_offset(int k, int kk, int K, int at) { return k < K - kk * kGemmStep ? at : kNoRead; }

}  // namespace t5a
