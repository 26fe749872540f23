// Device-side MXFP4 quantiser: fp32 or bf16 rows -> packed E2M1 codes + E8M0 scales, the operand
// format the GEMM kernels consume.  This is the step that precedes the GEMM in an MLP (the
// reference has no counterpart; the benchmark's synthetic operands were so far quantised with
// torch ops).  HBM-bound: every input element is read once, 0.53 bytes per element are written.
//
// Recipe (identical to the CPU oracle's quantize_mxfp4): per 32 consecutive k,
//   scale = 2^(floor(log2(amax)) - 2), exponent clamped to [-127, 127], stored as E8M0;
//   an all-zero block gets scale byte 127 and zero codes;
//   a block that holds an infinity or a NaN gets scale byte 0xFF (the E8M0 NaN) and zero codes;
//   elements are divided by the scale and rounded to nearest-even onto the E2M1 grid, saturating.
//
// Four lanes share a block, 8 consecutive elements each (eight lanes with 4 for large fp32 inputs, so that a load
// instruction reads whole consecutive lines); the block amax is formed with cross-lane exchanges.  The division and rounding are
// done by v_cvt_scalef32_pk_fp4_f32, whose scale operand contributes only its exponent.
#include "fp4_common.hpp"
#include "kernels.hpp"

namespace ave {
namespace {

// A piece of E elements of a block: amax over the 32 / E lanes that share the block, scale byte, codes.
template <int E>
__device__ inline void quantize_piece(const float (&v)[8], size_t i, uint8_t* packed, uint8_t* scales) {
  unsigned amax = lane_xor_max_bits(lane_xor_max_bits(abs_max_bits(v), 1), 2);
  if constexpr (E == 4) amax = lane_xor_max_bits(amax, 4);
  const int byte = mx_scale_byte(amax);
  const float scale = mx_scale_value(byte);
  unsigned codes = 0;
  codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, v[0], v[1], scale, 0);
  codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, v[2], v[3], scale, 1);
  if constexpr (E == 8) {
    codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, v[4], v[5], scale, 2);
    codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, v[6], v[7], scale, 3);
  }
  if (byte == 0xFF) codes = 0u;   // a block with an infinity or a NaN
  if constexpr (E == 8) reinterpret_cast<unsigned*>(packed)[i] = codes;
  else reinterpret_cast<uint16_t*>(packed)[i] = (uint16_t)codes;
  if (i % (32 / E) == 0) scales[i / (32 / E)] = (uint8_t)byte;
}

// T = float or __bf16.  A workgroup takes 256 U consecutive pieces of E elements per trip (one trip up to 2^20 workgroups), a lane
// U of them, 256 apart, with all its loads issued before the first use.  Bound by HBM; what counts is that the lines of a
// workgroup are neighbours and that inputs which no cache can hold do not pass through as if one could (NT):
// 14336 x 4096 fp32 51.5 us with trips over the whole tensor (5.2 TB/s, a copy: 4.9), 45.6 with consecutive pieces,
// 42.3 with NT and whole-line loads (6.3 TB/s); 4096 x 14336 bf16 27.9 -> 26.0.
// PAD: the output rows are laid out for row_pieces_out * E elements, more than the row_pieces_in * E that x has; the
// blocks behind a row's end are written as blocks of zeros (zero codes under the scale 2^0), which add nothing to a
// GEMM over the padded length.  n_blocks counts the OUTPUT blocks.
template <typename T, int E, int U, bool NT, bool PAD>
__global__ __launch_bounds__(256) void quantize_mx_kernel(const T* __restrict__ x, uint8_t* __restrict__ packed,
                                                          uint8_t* __restrict__ scales, size_t n_blocks,
                                                          unsigned row_pieces_in, unsigned row_pieces_out) {
  static_assert(E == 8 || (E == 4 && sizeof(T) == 4), "16 bytes a load");
  constexpr int V = E * (int)sizeof(T) / 16;   // loads of a piece
  const size_t pieces = n_blocks * (32 / E);   // trips start at multiples of 256: the lanes of a block stay together
  for (size_t i0 = (size_t)blockIdx.x * (256 * U) + threadIdx.x; i0 < pieces; i0 += (size_t)gridDim.x * (256 * U)) {
    v4i raw[U][V];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const size_t i = i0 + u * 256;
      size_t in = i;                 // the piece of x that output piece i is made from
      bool real = i < pieces;
      if constexpr (PAD) {
        const size_t row = i / row_pieces_out;
        const unsigned col = (unsigned)(i - row * row_pieces_out);
        real = real && col < row_pieces_in;
        in = row * row_pieces_in + col;
      }
#pragma unroll
      for (int q = 0; q < V; ++q) {
        raw[u][q] = v4i{0, 0, 0, 0};
        const v4i* src = reinterpret_cast<const v4i*>(x) + in * V + q;
        if (real) raw[u][q] = NT ? __builtin_nontemporal_load(src) : *src;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const size_t i = i0 + u * 256;
      float v[8] = {};
#pragma unroll
      for (int j = 0; j < E; ++j) {
        if constexpr (sizeof(T) == 4) {
          v[j] = __builtin_bit_cast(float, (int)raw[u][j / 4][j % 4]);
        } else {
          const unsigned pair = (unsigned)raw[u][0][j / 2];
          v[j] = __builtin_bit_cast(float, j % 2 ? pair & 0xFFFF0000u : pair << 16);
        }
      }
      if (i < pieces) quantize_piece<E>(v, i, packed, scales);   // uniform over the lanes of a block
    }
  }
}

template <typename T, int E, int U, bool NT>
hipError_t launch_form(const void* x, uint8_t* packed, uint8_t* scales, size_t n_blocks, int k, int k_padded, hipStream_t s) {
  const size_t trip = 256 * U;
  size_t grid = (n_blocks * (32 / E) + trip - 1) / trip;
  if (grid > 1u << 20) grid = 1u << 20;
  if (k_padded == k)
    hipLaunchKernelGGL((quantize_mx_kernel<T, E, U, NT, false>), dim3((unsigned)grid), dim3(256), 0, s,
                       static_cast<const T*>(x), packed, scales, n_blocks, 0u, 0u);
  else
    hipLaunchKernelGGL((quantize_mx_kernel<T, E, U, NT, true>), dim3((unsigned)grid), dim3(256), 0, s,
                       static_cast<const T*>(x), packed, scales, n_blocks, (unsigned)(k / E), (unsigned)(k_padded / E));
  return hipGetLastError();
}

template <typename T>
hipError_t launch(const void* x, uint8_t* packed, uint8_t* scales, size_t rows, int k, int k_padded, hipStream_t s) {
  const size_t n_blocks = rows * (size_t)(k_padded / 32);
  if (n_blocks == 0) return hipSuccess;
  // Above the 32 MB that the L2s hold together the input is streamed.  Below, and found in the caches, eight elements a lane
  // are the better form for fp32 (2048 x 4096: 5.7 us against 5.9), and NT makes no difference for bf16.
  const bool streamed = rows * (size_t)k * sizeof(T) > (32u << 20);
  if constexpr (sizeof(T) == 4)
    return streamed ? launch_form<T, 4, 2, true>(x, packed, scales, n_blocks, k, k_padded, s)
                    : launch_form<T, 8, 1, false>(x, packed, scales, n_blocks, k, k_padded, s);
  else if (n_blocks <= (1u << 15))   // a decode batch (1 M elements): one piece a lane keeps twice the compute units busy, 2.7 us against 2.8
    return launch_form<T, 8, 1, false>(x, packed, scales, n_blocks, k, k_padded, s);
  else
    return streamed ? launch_form<T, 8, 2, true>(x, packed, scales, n_blocks, k, k_padded, s)
                    : launch_form<T, 8, 2, false>(x, packed, scales, n_blocks, k, k_padded, s);
}

}  // namespace

hipError_t launch_quantize_mx(const void* x, int is_bf16, uint8_t* packed, uint8_t* scales, size_t rows, int k,
                              int k_padded, hipStream_t s) {
  return is_bf16 ? launch<__bf16>(x, packed, scales, rows, k, k_padded, s)
                 : launch<float>(x, packed, scales, rows, k, k_padded, s);
}

}  // namespace ave
