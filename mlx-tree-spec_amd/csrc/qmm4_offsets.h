// Byte offsets of the activation loads that may lie past the end of x, for the kernels that take them
// through raw buffer resources, and for the host test that checks them (tests/load_offsets.cpp).
//
// Rule of every buffer load here that must read nothing (a row past M, a phase past the range): its
// LANE offset lies at or past the buffer's size, and its scalar offset is one that a load inside the
// buffer has (0 where there is none). The compiler documents the scalar offset of the raw buffer
// builtins as excluded from bounds checking; the gfx9 ISA compares the lane offset with the size less
// the scalar offset. Under the first a row step kept in the scalar offset is not checked at all, under
// the second a scalar offset past the size leaves no defined difference: so rows step in the lane
// offset, and only the position within a row (the same for every row) is scalar.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qmm4 {

struct LoadOffset {
  uint32_t lane, scalar;
};

// Row-phase x staging: phases of 128 V values of k, `threads` threads per load pass, each row's run of a
// phase in kXC = 16 V pieces of 16 bytes. Thread tid's piece in pass j is slot tid % kXC of row m =
// tid / kXC + (threads / kXC) j, which holds piece (tid % kXC) ^ (m % 16). The part that holds for every
// pass (x in buffers below 2 GiB: `live` false goes to 2 GiB, and a row step more stays below 4 GiB):
template <int V, int THREADS>
__host__ __device__ inline uint32_t rowphase_x_base(int tid, int K) {
  constexpr int kXC = 16 * V;
  const int m = tid / kXC;
  return (uint32_t)m * (uint32_t)K * 2u + (uint32_t)(16 * ((tid % kXC) ^ m));
}
// Pass j of phase ph, base as above. With 8 rows per pass bit 3 of the row is j's: its XOR flips bit 7
// of the offset, which is the piece's (K % 512 == 0 then, so a row's start has bit 7 clear).
template <int V, int THREADS>
__host__ __device__ inline LoadOffset rowphase_x_offset(uint32_t base, int j, int ph, int K, bool live) {
  constexpr int kRows = THREADS / (16 * V);
  static_assert(kRows == 16 || kRows == 8, "rows per load pass");
  const uint32_t o = live ? base ^ (uint32_t)((j * kRows & 8) * 16) : 0x80000000u;
  return {o + (uint32_t)(j * kRows) * (uint32_t)K * 2u, live ? (uint32_t)(ph * 256 * V) : 0u};
}

// General kernel, x in units of 64 k: load i takes 8 rows, lane / 8 the row and lane % 8 its 16-byte piece,
// from row m0. Lane part of load i (x with 64 rows more below 2 GiB); u: the unit.
__host__ __device__ inline uint32_t general_x_base(int m0, int lane, int K) {
  return (uint32_t)(m0 + (lane >> 3)) * (uint32_t)K * 2u + (uint32_t)(lane & 7) * 16u;
}
__host__ __device__ inline LoadOffset general_x_offset(uint32_t base, int i, int u, int K, bool live) {
  return {live ? base + (uint32_t)i * 16u * (uint32_t)K : 0x80000000u, live ? (uint32_t)(u * 128) : 0u};
}

// GEMM activations: load pass j of RPP rows each, row r0 + RPP j of the tile at row m0, 16-byte chunk kc of
// K step kt (64 k). The lane part of pass 0, and the offset of pass j (x with 256 rows more below 4 GiB):
__host__ __device__ inline uint32_t gemm_x_base(int m0, int r0, int K, int kc) {
  return (uint32_t)(m0 + r0) * (uint32_t)K * 2u + (uint32_t)kc * 16u;
}
template <int RPP>
__host__ __device__ inline LoadOffset gemm_x_offset(uint32_t base, int j, int K, int kt) {
  return {base + (uint32_t)(j * RPP) * (uint32_t)K * 2u, (uint32_t)(kt * 128)};
}

}  // namespace qmm4
