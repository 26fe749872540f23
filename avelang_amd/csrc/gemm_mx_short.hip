// MXFP4 GEMM for gfx950 for small calls: a short K and few tiles, where a launch is over before a ring of LDS buffers is full.
//
// Bound by latency: the launch, one trip to memory, a few MFMAs and the store.  So nothing is staged: a workgroup owns a 32 x 32
// block of C, each of its four waves a quarter of K (up to 512 elements), of which it requests ALL operands at once, straight into registers
// in MFMA order; the four sums meet in LDS and are added in the order of K.  Four waves a block rather than one, because a load
// instruction that touches 32 rows takes 32 cycles of its compute unit's address path: at 256 x 256 x 512 that alone is 1 us for a wave
// that owns all of K.  For the same reason the time grows with blocks x K, which is what limits the sizes (mx_short_preferred).
#include "fp4_common.hpp"
#include "kernels.hpp"
#include "tile_common.hpp"

namespace ave {
namespace {

constexpr int kSplit = 4;   // waves of a workgroup, which share K

// Scale bytes of S consecutive blocks as the bytes of one or two dwords
template <int S>
struct Scales {
  int v[(S + 3) / 4];
  __device__ void load(const uint8_t* at) {
    if constexpr (S == 1) v[0] = *at;
    else if constexpr (S == 2) v[0] = *reinterpret_cast<const uint16_t*>(at);
    else {
#pragma unroll
      for (int i = 0; i < S / 4; ++i) v[i] = reinterpret_cast<const int*>(at)[i];
    }
  }
};

// S: MFMAs of a wave; lane half h of wave w multiplies blocks (2 w + h) S .. + S - 1 of 32 elements.  WHOLE: K = 256 S and scale
// rows that start at multiples of S (4 at most) bytes; otherwise a block behind the row's end is zeros under 2^0.
template <int S, bool WHOLE>
__global__ __launch_bounds__(kSplit * 64) void mx_short_kernel(MxArgs p, unsigned m_tiles) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int rho = lane & 31, h = lane >> 5;
  const int m0 = (int)(blockIdx.x % m_tiles) * 32, n0 = (int)(blockIdx.x / m_tiles) * 32;
  const int m = m0 + rho < p.M ? m0 + rho : p.M - 1;
  const int nn = n0 + pi_row(rho), n = nn < p.N ? nn : p.N - 1;
  const int blocks = p.K / kMxBlock, first = (2 * w + h) * S;
  const uint8_t* a_row = p.A + (size_t)m * (size_t)(p.K / 2);
  const uint8_t* b_row = p.B + (size_t)n * (size_t)(p.K / 2);
  const uint8_t* as_row = p.As + (size_t)m * (size_t)blocks;
  const uint8_t* bs_row = p.Bs + (size_t)n * (size_t)blocks;
  v4i a[S], b[S];
  v16f acc = {};
  if constexpr (WHOLE) {
    Scales<S> as, bs;
    as.load(as_row + first);
    bs.load(bs_row + first);
#pragma unroll
    for (int i = 0; i < S; ++i) {
      a[i] = *reinterpret_cast<const v4i*>(a_row + (first + i) * 16);
      b[i] = *reinterpret_cast<const v4i*>(b_row + (first + i) * 16);
    }
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int sa = as.v[i / 4], sb = bs.v[i / 4];
      if (i % 4 == 0) acc = mfma32<0, 0>(b[i], a[i], acc, sb, sa);
      else if (i % 4 == 1) acc = mfma32<1, 1>(b[i], a[i], acc, sb, sa);
      else if (i % 4 == 2) acc = mfma32<2, 2>(b[i], a[i], acc, sb, sa);
      else acc = mfma32<3, 3>(b[i], a[i], acc, sb, sa);
    }
  } else {
    int as[S], bs[S];
#pragma unroll
    for (int i = 0; i < S; ++i) {   // (a clamped address rather than a branch: every load goes out before the first is waited for)
      const int block = first + i < blocks ? first + i : blocks - 1;
      a[i] = *reinterpret_cast<const v4i*>(a_row + block * 16);
      b[i] = *reinterpret_cast<const v4i*>(b_row + block * 16);
      as[i] = as_row[block];
      bs[i] = bs_row[block];
    }
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const bool have = first + i < blocks;
      const v4i none = {0, 0, 0, 0};
      acc = mfma32<0, 0>(have ? b[i] : none, have ? a[i] : none, acc, have ? bs[i] : 127, have ? as[i] : 127);
    }
  }
  // wave w adds up registers 4 w .. 4 w + 3 of all waves and stores these four columns of every row
  __shared__ v4f sums[kSplit][4][64];
#pragma unroll
  for (int r = 0; r < 4; ++r) sums[w][r][lane] = v4f{acc[4 * r], acc[4 * r + 1], acc[4 * r + 2], acc[4 * r + 3]};
  __syncthreads();
  v4f d = sums[0][w][lane];
#pragma unroll
  for (int k = 1; k < kSplit; ++k) d += sums[k][w][lane];
  const int row = m0 + rho, col = n0 + 16 * (w >> 1) + 8 * h + 4 * (w & 1);
  if (row >= p.M) return;
  uint16_t* c = p.C + (size_t)row * p.N + col;
  const v2i o = {(int)pack_bf16x2(d[0], d[1]), (int)pack_bf16x2(d[2], d[3])};
  if (col + 4 <= p.N && p.N % 4 == 0 && (reinterpret_cast<uintptr_t>(p.C) & 7) == 0) {
    *reinterpret_cast<v2i*>(c) = o;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col + e < p.N) c[e] = (uint16_t)(((unsigned)o[e >> 1] >> (16 * (e & 1))) & 0xFFFF);
  }
}

template <int S>
hipError_t launch(const MxArgs& p, hipStream_t s) {
  const unsigned m_tiles = ((unsigned)p.M + 31) / 32, n_tiles = ((unsigned)p.N + 31) / 32;
  const uintptr_t at = reinterpret_cast<uintptr_t>(p.As) | reinterpret_cast<uintptr_t>(p.Bs);
  const bool whole = p.K == 256 * S && at % (S < 4 ? S : 4) == 0;
  if (whole) hipLaunchKernelGGL((mx_short_kernel<S, true>), dim3(m_tiles * n_tiles), dim3(kSplit * 64), 0, s, p, m_tiles);
  else hipLaunchKernelGGL((mx_short_kernel<S, false>), dim3(m_tiles * n_tiles), dim3(kSplit * 64), 0, s, p, m_tiles);
  return hipGetLastError();
}

}  // namespace

// the plain GEMM, K up to 2048 (a multiple of 32), 16-byte aligned A and B, a tile count that fits an int
bool mx_short_supports(const MxArgs& p) {
  if (p.row_offsets || p.swiglu || p.blocked_scales || p.M <= 0 || p.N <= 0 || p.K <= 0 || p.K > 2048 || p.K % kMxBlock != 0) return false;
  if (((reinterpret_cast<uintptr_t>(p.A) | reinterpret_cast<uintptr_t>(p.B)) & 15) != 0) return false;
  return ((uint64_t)p.M + 31) / 32 * (((uint64_t)p.N + 31) / 32) < (1ull << 23);
}

// Shape-based dispatch, from graph replays of 430 shapes (K 64 .. 2048, 1 .. 2048 rows, N 256 .. 16384).  In rounds of one 32 x 32 block per
// compute unit this kernel takes about 2.1 us + 0.4 (K = 256), 0.7 (512), 1.35 (1024) a round.  Against it, us before -> here:
//  * K below 512 that no 256 divides: the one-wave kernel (gemm_generic.hip) waits for every 64 elements: 600 x 2560 x 288 8.0 -> 4.6,
//    256 x 16384 x 160 13.6 -> 6.8, 8192 x 8192 x 480 227 -> 125;
//  * K = 256: the 256 x 256 kernel's tiles take 5.2 from 17 rows on: 256 x 256 x 256 5.3 -> 2.4, 600 x 2560 5.8 -> 4.4, equal at 8 rounds;
//  * K = 512 .. 1023: the ring kernels take 2.6 - 3.3 up to 32 rows, 5.4 - 9 up to 64, the narrow-tile kernel 4.0 - 5.2 above:
//    16 x 4096 x 512 2.8 -> 2.5, 64 x 8192 x 768 7.5 -> 4.4, 100 x 2560 x 768 5.1 -> 4.3, 256 x 4096 x 512 equal (4 rounds);
//  * K = 1024: 64 x 4096 3.7 -> 3.3, 256 x 1024 5.3 -> 3.3; up to 32 rows the rings are as fast;
//  * above: more than 64 rows and one round: 100 x 1024 x 2048 6.4 -> 4.6, 256 x 1024 x 1280 6.1 -> 4.8; two rounds 0.8 times as fast.
bool mx_short_preferred(int M, int N, int K, int cus) {
  if (M <= 0 || N <= 0 || K > 2048) return false;
  if (cus <= 0) cus = 256;
  const uint64_t tiles = ((uint64_t)M + 31) / 32 * (((uint64_t)N + 31) / 32);
  auto rounds_up_to = [&](int r) { return tiles <= (uint64_t)r * (uint64_t)cus; };
  if (K < 512 && K % 256 != 0) return tiles < (1ull << 23);
  if (K == 256) return rounds_up_to(M <= 16 ? 2 : 6);
  if (K < 1024) return rounds_up_to(M <= 32 ? 2 : (M <= 64 ? 4 : (K == 512 ? 3 : 2)));
  if (K == 1024) return M > 32 && rounds_up_to(M <= 64 ? 1 : 2);
  return M > 64 && rounds_up_to(1);
}

hipError_t launch_mx_short(const MxArgs& p, hipStream_t s) {
  if (p.K <= 256) return launch<1>(p, s);
  if (p.K <= 512) return launch<2>(p, s);
  if (p.K <= 1024) return launch<4>(p, s);
  return launch<8>(p, s);
}

}  // namespace ave
