// Quantized matmul in the formats and shapes the packed kernels do not take: y = x @ dequant(w)^T for
// 2-, 4- or 8-bit codes in groups of 32, 64 or 128, any number of columns, K % 64 == 0 (what the
// reference hands to MLX's own op, src/mlx_tree_spec/packed_linear.py:56-57, 84-86). The weights are
// dequantized in registers, bit for bit as dequantize() does (bf16_rne(fp32(s) * q + fp32(b))), and
// multiplied on bf16 MFMA with fp32 accumulation.
//
//  * A workgroup (8 waves) computes 16 CB columns of 16 MB rows over the whole of K; its waves split
//    K into 8 contiguous slices and share nothing until the end, so the loop has no barrier. Splitting
//    K over the waves keeps every column block's weights in one workgroup (no partial sums in memory)
//    and still gives small N 8 waves per 16 columns.
//  * A wave walks its slice in units of 64 k, the loads of the next unit in flight. Lane (n, g) = (lane
//    % 16, lane / 16) loads the codes of k = 16 g .. 16 g + 15 of weight row n (16, 8 or 4 bytes): the
//    B operands of two MFMA 16x16x32, whose A operand holds the same k of x.
//  * x is loaded 8 rows x 128 bytes per instruction (neighbouring lanes in one row, which the address
//    unit merges) and put in A-fragment order through the wave's own LDS (pieces XOR-swizzled by
//    row / 2, so that the 16 rows of one read fall in distinct banks). The scales and biases of 8
//    units are loaded together, four neighbouring lanes per row, through that LDS too.
//  * The waves' sums are added in wave order (deterministic), one f32x4 per thread.
// Bound: launch and memory latency at small sizes, x from L2 (each workgroup reads its rows of x
// whole) and the dequantization VALU past that. Against the dequantization kernel and a library
// product of its bf16 weights (GPU time by events, which the host bounds below ~29 us there): 24 x 2560
// -> 4100 8-bit groups of 32 29.6 -> 7.2 us (a streaming read of its 11.8 MB 3.5), 2 x 8192 -> 8191
// 8-bit 65.8 -> 16.8, 64 x 8192 -> 8191 8-bit 80.8 -> 28.5, 256 x 8192 -> 8191 8-bit 136.9 -> 90.4.
#include "qmm4_common.h"
#include "qmm4_kernels.h"
#include "qmm4_offsets.h"

namespace qmm4 {

namespace {

constexpr int kGnWaves = 8;
constexpr int kGnSeg = 8;     // units per scale segment
constexpr int kGnScMax = 16;  // groups of a segment (8 units of 64 k in groups of 32)
constexpr int kGnScPitch = kGnScMax + 2;  // bf16 per row in LDS

struct GeneralParams {
  const uint16_t* x;
  const uint32_t* w;
  const uint16_t* s;
  const uint16_t* b;
  uint16_t* y;
  int M, N, K;
  int gshift;  // log2 of the group size
};

template <int BITS>
struct Codes;  // 16 codes of one weight row
template <>
struct Codes<8> { u32x4 v; };
template <>
struct Codes<4> { u32x2 v; };
template <>
struct Codes<2> { uint32_t v; };

// B operand of MFMA t: codes 8 t .. 8 t + 7.
__device__ __forceinline__ u32x4 dequant8(const Codes<8>& c, int t, float s, float b) {
  u32x4 r;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t d = c.v[2 * t + h];
    r[2 * h] = pack_bf16x2(__builtin_fmaf((float)(d & 0xFFu), s, b), __builtin_fmaf((float)((d >> 8) & 0xFFu), s, b));
    r[2 * h + 1] = pack_bf16x2(__builtin_fmaf((float)((d >> 16) & 0xFFu), s, b), __builtin_fmaf((float)(d >> 24), s, b));
  }
  return r;
}
__device__ __forceinline__ u32x4 dequant8(const Codes<4>& c, int t, float s, float b) {
  return dequant_word(c.v[t], s, s * 0.0625f, b);
}
__device__ __forceinline__ u32x4 dequant8(const Codes<2>& c, int t, float s, float b) {
  u32x4 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int o = 16 * t + 4 * j;
    r[j] = pack_bf16x2(__builtin_fmaf((float)((c.v >> o) & 3u), s, b), __builtin_fmaf((float)((c.v >> (o + 2)) & 3u), s, b));
  }
  return r;
}

template <int MB, int CB>
struct GnCfg {
  static constexpr int NX = 2 * MB;  // x loads per unit (8 rows each)
  static constexpr size_t kXBytes = (size_t)16 * MB * 128;
  static constexpr size_t kScBytes = (size_t)CB * 2 * 16 * kGnScPitch * 2;
  static constexpr size_t kMain = kGnWaves * (kXBytes + kScBytes);
  static constexpr size_t kRed = (size_t)kGnWaves * MB * CB * 64 * 16;
  static constexpr size_t kLds = kMain > kRed ? kMain : kRed;
  static_assert(MB * CB * 64 <= 64 * kGnWaves, "one sum per thread");
  static_assert(kScBytes % 16 == 0, "aligned");
};

template <int BITS, int MB, int CB>
__global__ __launch_bounds__(64 * kGnWaves) __attribute__((amdgpu_waves_per_eu(2)))
void general_kernel(GeneralParams P) {
  using C = GnCfg<MB, CB>;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int m0 = blockIdx.y * 16 * MB, c0 = blockIdx.x * 16 * CB;
  const int U = P.K >> 6;
  const int ub = (int)((long long)wave * U / kGnWaves), ue = (int)((long long)(wave + 1) * U / kGnWaves);
  const int KG = P.K >> P.gshift;
  const int wrow = P.K / 8 * BITS;  // bytes of a weight row

  // Rows past M, columns past N and groups past the last row lie past the end of their buffers (each
  // below 2 GiB) by their lane offsets and read as zero; kOut is past the end of all of them.
  constexpr uint32_t kOut = 0x80000000u;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(P.x), 0, rsrc_bytes((unsigned long long)P.M * P.K * 2), kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(P.w), 0, rsrc_bytes((unsigned long long)P.N * wrow), kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(P.s), 0, rsrc_bytes((unsigned long long)P.N * KG * 2), kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(P.b), 0, rsrc_bytes((unsigned long long)P.N * KG * 2), kBufferRsrcWord3);

  u32x4* const xl = reinterpret_cast<u32x4*>(lds + (size_t)wave * (C::kXBytes + C::kScBytes));
  uint16_t* const sl = reinterpret_cast<uint16_t*>(lds + (size_t)wave * (C::kXBytes + C::kScBytes) + C::kXBytes);

  u32x4 xr[2][C::NX];
  Codes<BITS> wr[2][CB];
  const uint32_t xo = general_x_base(m0, lane, P.K);
  auto load = [&](int j, int u) __attribute__((always_inline)) {
    const bool live = u < ue;
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      const uint32_t o = live ? (uint32_t)(c0 + 16 * c + n) * (uint32_t)wrow + (uint32_t)(g * 2 * BITS) : kOut;
      const int so = live ? u * 8 * BITS : 0;
      if constexpr (BITS == 8) wr[j][c].v = __builtin_amdgcn_raw_buffer_load_b128(rw, o, so, 0);
      if constexpr (BITS == 4) wr[j][c].v = __builtin_amdgcn_raw_buffer_load_b64(rw, o, so, 0);
      if constexpr (BITS == 2) wr[j][c].v = __builtin_amdgcn_raw_buffer_load_b32(rw, o, so, 0);
    }
#pragma unroll
    for (int i = 0; i < C::NX; ++i) {
      const LoadOffset xi = general_x_offset(xo, i, u, P.K, live);
      xr[j][i] = __builtin_amdgcn_raw_buffer_load_b128(rx, xi.lane, (int)xi.scalar, 0);
    }
  };
  // Scales and biases of the segment from unit u: groups g0 + lane % 4 + 4 j of row lane / 4.
  constexpr int kNL = kGnScMax / 4;
  uint16_t sr[CB][2][kNL];
  const int nl = P.gshift == 5 ? 4 : 2;  // 16 groups of 32, 8 of 64, up to 5 of 128
  auto load_sc = [&](int u) __attribute__((always_inline)) {
    const int g0 = (u * 64) >> P.gshift;
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int j = 0; j < kNL; ++j) {
        const int gr = g0 + (lane & 3) + 4 * j;
        const uint32_t o =
            u < ue && j < nl ? ((uint32_t)(c0 + 16 * c + (lane >> 2)) * (uint32_t)KG + (uint32_t)gr) * 2u : kOut;
        sr[c][0][j] = __builtin_amdgcn_raw_buffer_load_b16(rs, o, 0, 0);
        sr[c][1][j] = __builtin_amdgcn_raw_buffer_load_b16(rb, o, 0, 0);
      }
  };
  // Data that the lanes of a wave hand to each other through the wave's own LDS needs no barrier (a
  // wave's LDS accesses complete in order), but the compiler, which sees one lane, must keep the order.
  auto lds_order = [&]() __attribute__((always_inline)) { asm volatile("" ::: "memory"); };
  auto put_sc = [&]() __attribute__((always_inline)) {
    lds_order();
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int j = 0; j < kNL; ++j)
          sl[((c * 2 + a) * 16 + (lane >> 2)) * kGnScPitch + (lane & 3) + 4 * j] = sr[c][a][j];
    lds_order();
  };

  f32x4 acc[MB][CB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int c = 0; c < CB; ++c) acc[i][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  auto compute = [&](int j, int u, int g0) __attribute__((always_inline)) {
    lds_order();
#pragma unroll
    for (int i = 0; i < C::NX; ++i) {
      const int m = 8 * i + (lane >> 3);
      xl[m * 8 + ((lane & 7) ^ ((m >> 1) & 7))] = xr[j][i];
    }
    lds_order();
    const int gi = ((u * 64 + 16 * g) >> P.gshift) - g0;
    float sf[CB], bf[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      sf[c] = bf16_to_f32(sl[((c * 2) * 16 + n) * kGnScPitch + gi]);
      bf[c] = bf16_to_f32(sl[((c * 2 + 1) * 16 + n) * kGnScPitch + gi]);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      u32x4 a[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i) a[i] = xl[(16 * i + n) * 8 + ((2 * g + t) ^ ((n >> 1) & 7))];
#pragma unroll
      for (int c = 0; c < CB; ++c) {
        const u32x4 B = dequant8(wr[j][c], t, sf[c], bf[c]);
#pragma unroll
        for (int i = 0; i < MB; ++i)
          acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[i]), as_bf16x8(B), acc[i][c], 0, 0, 0);
      }
    }
  };

  load_sc(ub);
  load(0, ub);
  for (int seg = ub; seg < ue; seg += kGnSeg) {
    const int g0 = (seg * 64) >> P.gshift;
    const int se = min(seg + kGnSeg, ue);
    put_sc();
    load_sc(seg + kGnSeg);
    int u = seg;
    for (; u + 2 <= se; u += 2) {
      load(1, u + 1);
      compute(0, u, g0);
      load(0, u + 2);
      compute(1, u + 1, g0);
    }
    if (u < se) compute(0, u, g0);  // an odd count ends the wave's slice (segments are of even length)
  }

  __syncthreads();  // the sums take the place of x
  f32x4* const red = reinterpret_cast<f32x4*>(lds);
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int c = 0; c < CB; ++c) red[((wave * MB + i) * CB + c) * 64 + lane] = acc[i][c];
  __syncthreads();
  if (tid >= MB * CB * 64) return;
  f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int q = 0; q < kGnWaves; ++q) {
    const f32x4 v = red[q * (MB * CB * 64) + tid];
    sum[0] += v[0]; sum[1] += v[1]; sum[2] += v[2]; sum[3] += v[3];
  }
  const int c = wave % CB, i = wave / CB;
  const int col = c0 + 16 * c + n;
  if (col >= P.N) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int m = m0 + 16 * i + 4 * g + r;
    if (m < P.M) P.y[(size_t)m * P.N + col] = (uint16_t)bf16_rne(sum[r]);
  }
}

template <int BITS, int MB, int CB>
hipError_t launch_general_t(const GeneralParams& P, hipStream_t stream) {
  using C = GnCfg<MB, CB>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&general_kernel<BITS, MB, CB>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::kLds);
  if (e != hipSuccess) return e;
  const dim3 grid((unsigned)((P.N + 16 * CB - 1) / (16 * CB)), (unsigned)((P.M + 16 * MB - 1) / (16 * MB)));
  hipLaunchKernelGGL((general_kernel<BITS, MB, CB>), grid, dim3(64 * kGnWaves), C::kLds, stream, P);
  return hipGetLastError();
}

// Two column blocks per wave (x read half as often, and each A fragment feeds two MFMAs) when the grid
// then still has a workgroup per CU, or past 16 rows (more x per weight) one per two CUs. One / two
// blocks: 24 x 2560 -> 4100 8-bit (129 workgroups of two) 7.7 / 7.2 us, 64 x 8192 -> 8191 8-bit 40.4 /
// 28.5, 7 x 8192 -> 8191 4-bit 17.0 / 15.0, but 1 x 2560 -> 4100 8-bit 5.5 / 5.9 and 40 x 8192 -> 513 (17
// workgroups) 14.8 / 20.3.
template <int BITS>
hipError_t launch_general_b(const GeneralParams& P, int cus, hipStream_t stream) {
  const long long wgs = (long long)((P.N + 31) / 32) * ((P.M + 63) / 64);
  const bool two = P.M <= 16 ? wgs >= cus : 2 * wgs >= cus;
  if (P.M <= 16) return two ? launch_general_t<BITS, 1, 2>(P, stream) : launch_general_t<BITS, 1, 1>(P, stream);
  if (P.M <= 32) return two ? launch_general_t<BITS, 2, 2>(P, stream) : launch_general_t<BITS, 2, 1>(P, stream);
  return two ? launch_general_t<BITS, 4, 2>(P, stream) : launch_general_t<BITS, 4, 1>(P, stream);
}

}  // namespace

hipError_t launch_general(const uint16_t* x, const uint32_t* w, const uint16_t* s, const uint16_t* b, uint16_t* y,
                          int M, int N, int K, int group_size, int bits, int cus, hipStream_t stream) {
  GeneralParams P;
  P.x = x; P.w = w; P.s = s; P.b = b; P.y = y;
  P.M = M; P.N = N; P.K = K;
  P.gshift = group_size == 32 ? 5 : group_size == 64 ? 6 : group_size == 128 ? 7 : -1;
  if (P.gshift < 0 || K % 64 != 0 || K % group_size != 0) return hipErrorInvalidValue;
  switch (bits) {
    case 2: return launch_general_b<2>(P, cus, stream);
    case 4: return launch_general_b<4>(P, cus, stream);
    case 8: return launch_general_b<8>(P, cus, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace qmm4
