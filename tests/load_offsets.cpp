// Host-only check of the activation loads' buffer offsets (csrc/qmm4_offsets.h): for every thread, pass
// and position of a kernel's walk, a load of a row below M reads that row's bytes, and a load of any
// other row, or of a phase past the range, is dropped by the buffer's bounds check, whether that check
// leaves the scalar offset out (as the compiler documents its builtins) or compares the lane offset
// with the size less the scalar offset in 32 bits (the gfx9 ISA). Prints one line per violation and a
// summary; the exit status is 1 if there was one. Built and run by tests/test_load_offsets.py.
#include <cstdio>
#include <cstring>

#include "qmm4_offsets.h"

using namespace qmm4;

namespace {

long long g_fail = 0, g_checked = 0;

// A 16-byte load at `o` of a buffer of `size` bytes: `want` is the byte it must read from, or -1 for
// none.
void check(const char* what, const LoadOffset& o, uint32_t size, long long want, int M, int K, int a, int b) {
  ++g_checked;
  const bool drop_lane = o.lane >= size;                    // scalar offset not compared
  const bool drop_isa = o.lane >= (uint32_t)(size - o.scalar);  // scalar offset taken from the size
  const long long at = (long long)o.lane + o.scalar;
  const bool ok = want < 0 ? drop_lane && drop_isa : !drop_lane && !drop_isa && at == want && at + 16 <= (long long)size;
  if (ok) return;
  if (g_fail++ < 20)
    std::printf("FAIL %s M=%d K=%d (%d, %d): lane %u scalar %u of %u bytes, wanted %lld\n", what, M, K, a, b, o.lane,
                o.scalar, size, want);
}

template <int V, int MP>
void rowphase(int M, int K) {
  constexpr int kThreads = 512, kXC = 16 * V, kRows = kThreads / kXC;
  const int NP = K / (128 * V);
  const uint32_t size = (uint32_t)M * K * 2u;
  for (int tid = 0; tid < kThreads; ++tid) {
    const uint32_t base = rowphase_x_base<V, kThreads>(tid, K);
    for (int j = 0; j < MP / kRows; ++j) {
      const int m = tid / kXC + kRows * j;
      for (int ph = 0; ph < NP + 2; ++ph) {  // prefetches run two phases past the last
        const bool live = ph < NP;
        const long long want =
            live && m < M ? (long long)m * K * 2 + ph * 256 * V + 16 * ((tid % kXC) ^ (m % 16)) : -1;
        check("rowphase", rowphase_x_offset<V, kThreads>(base, j, ph, K, live), size, want, M, K, tid, j);
      }
    }
  }
}

template <int MP>
void rowphase_rows() {
  for (int M : {MP > 64 ? MP - 15 : MP / 2 + 1, MP - 1, MP}) {
    for (int K : {512, 1024, 5120}) {
      rowphase<2, MP>(M, K);
      if (MP <= 32) rowphase<4, MP <= 32 ? MP : 32>(M, K);
    }
  }
}

// The general kernel's x: MB row blocks of 16 from m0, units of 64 k and one past the slice's last.
template <int MB>
void general(int M, int K) {
  const uint32_t size = (uint32_t)M * K * 2u;
  for (int m0 = 0; m0 < M; m0 += 16 * MB)
    for (int lane = 0; lane < 64; ++lane) {
      const uint32_t base = general_x_base(m0, lane, K);
      for (int i = 0; i < 2 * MB; ++i)
        for (int u = 0; u <= K / 64; ++u) {
          const int m = m0 + 8 * i + lane / 8;
          const bool live = u < K / 64;
          const long long want = live && m < M ? (long long)m * K * 2 + u * 128 + lane % 8 * 16 : -1;
          check("general", general_x_offset(base, i, u, K, live), size, want, M, K, lane, i);
        }
    }
}

// The GEMM's activations: tiles of BM rows, RPP rows per load pass, K steps of 64.
template <int BM, int RPP>
void gemm(int M, int K) {
  const uint32_t size = (uint32_t)M * K * 2u;
  for (int m0 = 0; m0 < (M + 255) / 256 * 256; m0 += BM)  // quarters of a 256-row tile may lie past M whole
    for (int r0 = 0; r0 < RPP; ++r0)
      for (int kc = 0; kc < 8; ++kc)
        for (int j = 0; j < BM / RPP; ++j)
          for (int kt = 0; kt < K / 64; ++kt) {
            const int m = m0 + r0 + RPP * j;
            const long long want = m < M ? (long long)m * K * 2 + kt * 128 + kc * 16 : -1;
            check("gemm", gemm_x_offset<RPP>(gemm_x_base(m0, r0, K, kc), j, K, kt), size, want, M, K, r0, j);
          }
}

}  // namespace

int main() {
  rowphase<2, 16>(1, 512);
  rowphase<4, 16>(1, 512);
  rowphase_rows<16>();
  rowphase_rows<32>();
  rowphase_rows<64>();
  rowphase_rows<80>();
  rowphase_rows<96>();
  rowphase_rows<112>();
  rowphase_rows<128>();
  for (int K : {64, 192, 2560}) {
    for (int M : {1, 7, 8, 9, 16}) general<1>(M, K);
    for (int M : {17, 24, 25, 32}) general<2>(M, K);
    for (int M : {33, 64, 65, 100, 257}) general<4>(M, K);
  }
  for (int K : {128, 1024})
    for (int M : {65, 127, 128, 129, 203, 256, 300}) {
      gemm<128, 64>(M, K);
      gemm<256, 64>(M, K);
      gemm<256, 32>(M, K);  // the role-split kernel
    }
  std::printf("loads checked: %lld, violations: %lld\n", g_checked, g_fail);
  return g_fail ? 1 : 0;
}
