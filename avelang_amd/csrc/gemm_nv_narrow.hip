// NVFP4 GEMM for gfx950 on 128-column tiles: batches between the weight-streaming kernels' few rows and the prefill
// shapes that fill the chip with 256 x 256 tiles, and every K (a multiple of 16).
//
// Bound by the conversions (fp4 -> f16, see gemm_nv_tile.hip for why f16) and, with few rows, by the load path.  What
// decides how many conversions an MFMA costs is the shape of a WAVE's part of the tile -- a wave converts its own
// fragments: 64 x 64 takes 8 conversions-and-multiplies' worth of 16 k for every MFMA, 64 x 32 takes 12.  A 128 x 128 tile
// cut into eight parts would give every wave 64 x 32; here the eight waves are two groups of four 64 x 64 parts, and
// the groups take alternate 64-element groups of K (a 64 x 128 tile: four groups of two).  Their sums meet in LDS at the end.
//
// A stage is 256 elements of K; a ring of four (128 rows: 36 KB each) or five (64 rows: 27 KB) stage buffers is filled with
// global_load_lds_dwordx4, every wave loading an eighth of a stage, three stages ahead.  Layout, swizzle and K
// order inside a 64-element group are those of gemm_nv_tile.hip.  The pipeline runs across stages and the loop body has no branches:
// a stage's barrier sits at the start of its last group of steps, behind it every wave may read the next stage.
//
// K tail (K % 256): one more stage, whose loads are moved back so that they end where the row ends -- the last 16 scale
// bytes, and for K % 32 == 16 a last piece of codes that starts 8 bytes early -- because what lies behind the last row may
// not be memory.  Its fragments are put right (or zeroed) in registers before they are converted.
#include "fp4_common.hpp"
#include "kernels.hpp"
#include "tile_common.hpp"
#include "tile_map.hpp"

namespace ave {
namespace {

constexpr int BN = 128, BK = 256;
constexpr int kWaves = 8;
constexpr int kRowBytes = BK / 2;    // 128
constexpr int kScaleRow = BK / 16;   // 16 bytes

template <int WM>   // 64-row halves of a tile
struct Geo {
  static constexpr int kRows = 64 * WM;
  static constexpr int kOffB = kRows * kRowBytes;
  static constexpr int kOffS = kOffB + BN * kRowBytes;              // scale rows: A's, then B's
  static constexpr int kStage = kOffS + (kRows + BN) * kScaleRow;   // 36864 / 27648
  static constexpr int kRing = WM == 2 ? 4 : 5;
  static constexpr int kLds = kRing * kStage;                       // 147456 / 138240
  static constexpr int kLoads = WM + 3;                             // of one wave and stage: WM of A, 2 of B, 1 of scales
  static constexpr int kGroups = 4 / WM;                            // wave groups along K: 2 / 4
  static constexpr int kSteps = 16 / kGroups;                       // 16-element steps of a wave in a stage
};
static_assert(Geo<1>::kLds <= 160 * 1024 && Geo<2>::kLds <= 160 * 1024, "LDS of one compute unit");

// One wave's loads of a stage, skipped as a whole when `on` (a scalar) is 0: WM pieces of 8 rows of A to ma + 1024 i, two
// of B to mb + 1024 i, and 32 scale rows (lanes 0-31) to ms.
template <int WM>
__device__ inline void load_stage(int on, unsigned ma, unsigned mb, unsigned ms, const void* ga, const void* gb, const void* gs,
                                  const unsigned (&a)[2], const unsigned (&b)[2], unsigned sc) {
  unsigned long long saved;
  if constexpr (WM == 2)
    asm volatile(
        "s_cmp_eq_u32 %[on], 0\n\t"
        "s_cbranch_scc1 1f\n\t"
        "s_mov_b32 m0, %[ma]\n\t s_nop 0\n\t global_load_lds_dwordx4 %[a0], %[ga]\n\t"
        "s_mov_b32 m0, %[mb]\n\t s_nop 0\n\t global_load_lds_dwordx4 %[b0], %[gb]\n\t"
        "s_add_u32 m0, %[ma], 0x0400\n\t s_nop 0\n\t global_load_lds_dwordx4 %[a1], %[ga]\n\t"
        "s_add_u32 m0, %[mb], 0x0400\n\t s_nop 0\n\t global_load_lds_dwordx4 %[b1], %[gb]\n\t"
        "s_mov_b32 m0, %[ms]\n\t s_mov_b64 %[sv], exec\n\t s_mov_b32 exec_hi, 0\n\t global_load_lds_dwordx4 %[sc], %[gs]\n\t"
        "s_mov_b64 exec, %[sv]\n\t"
        "1:\n\t"
        : [sv] "=&s"(saved)
        : [on] "s"(on), [ma] "s"(ma), [mb] "s"(mb), [ms] "s"(ms), [ga] "s"(ga), [gb] "s"(gb), [gs] "s"(gs), [a0] "v"(a[0]),
          [a1] "v"(a[1]), [b0] "v"(b[0]), [b1] "v"(b[1]), [sc] "v"(sc)
        : "m0", "scc", "memory");
  else
    asm volatile(
        "s_cmp_eq_u32 %[on], 0\n\t"
        "s_cbranch_scc1 1f\n\t"
        "s_mov_b32 m0, %[ma]\n\t s_nop 0\n\t global_load_lds_dwordx4 %[a0], %[ga]\n\t"
        "s_mov_b32 m0, %[mb]\n\t s_nop 0\n\t global_load_lds_dwordx4 %[b0], %[gb]\n\t"
        "s_add_u32 m0, %[mb], 0x0400\n\t s_nop 0\n\t global_load_lds_dwordx4 %[b1], %[gb]\n\t"
        "s_mov_b32 m0, %[ms]\n\t s_mov_b64 %[sv], exec\n\t s_mov_b32 exec_hi, 0\n\t global_load_lds_dwordx4 %[sc], %[gs]\n\t"
        "s_mov_b64 exec, %[sv]\n\t"
        "1:\n\t"
        : [sv] "=&s"(saved)
        : [on] "s"(on), [ma] "s"(ma), [mb] "s"(mb), [ms] "s"(ms), [ga] "s"(ga), [gb] "s"(gb), [gs] "s"(gs), [a0] "v"(a[0]),
          [b0] "v"(b[0]), [b1] "v"(b[1]), [sc] "v"(sc)
        : "m0", "scc", "memory");
}

// Waits until at most `left` stages' loads (kLoads each) of this wave are outstanding; left is a scalar, 0 .. 2.
template <int LOADS>
__device__ inline void wait_stages(int left) {
  asm volatile(
      "s_cmp_ge_i32 %[l], 2\n\t"
      "s_cbranch_scc1 2f\n\t"
      "s_cmp_eq_u32 %[l], 1\n\t"
      "s_cbranch_scc1 1f\n\t"
      "s_waitcnt vmcnt(0)\n\t"
      "s_branch 3f\n\t"
      "1:\n\t"
      "s_waitcnt vmcnt(%[one])\n\t"
      "s_branch 3f\n\t"
      "2:\n\t"
      "s_waitcnt vmcnt(%[two])\n\t"
      "3:\n\t"
      :
      : [l] "s"(left), [one] "n"(LOADS), [two] "n"(2 * LOADS)
      : "scc", "memory");
}

__device__ inline int lds_read1(unsigned addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) unsigned char*>((uintptr_t)addr);
}
__device__ inline v4f lds_read16f(unsigned addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) v4f*>((uintptr_t)addr);
}
__device__ inline void lds_write16f(unsigned addr, v4f v) {
  *reinterpret_cast<__attribute__((address_space(3))) v4f*>((uintptr_t)addr) = v;
}

// SPLITK: workgroup pid is tile pid % tiles of K slice pid / tiles; a slice is p.slice_stages stages (the last one what
// is left, the K tail with it), its fp32 sums (times the two per-tensor scales) go to p.P[slice][M][N].
template <int WM, bool SPLITK>
__global__ __launch_bounds__(kWaves * 64) void nv_narrow_kernel(NvArgs p, int m_tiles, int n_tiles) {
  using G = Geo<WM>;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int wn = w & 1, wm = (w >> 1) % WM, kg = w / (2 * WM);

  int tm, tn, slice = 0;
  {
    int pid = blockIdx.x;
    if (SPLITK) {
      slice = pid / (m_tiles * n_tiles);
      pid -= slice * (m_tiles * n_tiles);
    }
    map_tile(pid, m_tiles, n_tiles, tm, tn);
  }
  const int m_begin = tm * G::kRows, n_begin = tn * BN;
  const unsigned row_bytes = (unsigned)p.K / 2, row_scales = (unsigned)p.K / 16;
  const int all_stages = p.K / BK, tail_blocks = (p.K % BK) / 16;   // whole stages; 16-element blocks behind them
  const int s_begin = SPLITK ? slice * p.slice_stages : 0;
  const int s_end = SPLITK && s_begin + p.slice_stages < all_stages ? s_begin + p.slice_stages : all_stages;
  const bool tail = tail_blocks != 0 && s_end == all_stages;
  const int stages = s_end - s_begin, loads = stages + (tail ? 1 : 0);   // stages to multiply in the loop; to load

  // ---- this wave's loads -------------------------------------------------------------------------------------------
  // A: tile rows (WM w + i) * 8 .. + 7; B: (2 w + i) * 8 .. + 7; lane -> (row, swizzled 16-byte chunk).  Scale rows: 32 of A for
  // waves below 2 WM, 32 of B for the next four; with 64-row tiles waves 6 and 7 repeat rows of wave 5.
  // Rows past the end of a matrix are clamped to its last row: their products land in elements of C never stored.
  unsigned a_off[2], b_off[2], s_off;
  int chunk_a[2], chunk_b[2];
  {
    const int lr = lane >> 3, cprime = lane & 7;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int ra = (WM * w + (i % WM)) * 8 + lr, rb = (2 * w + i) * 8 + lr;
      int am = m_begin + ra, bn = n_begin + rb;
      am = am < p.M ? am : p.M - 1;
      bn = bn < p.N ? bn : p.N - 1;
      chunk_a[i] = cprime ^ ((ra >> 1) & 7);
      chunk_b[i] = cprime ^ ((rb >> 1) & 7);
      a_off[i] = (unsigned)am * row_bytes + chunk_a[i] * 16;
      b_off[i] = (unsigned)bn * row_bytes + chunk_b[i] * 16;
    }
  }
  const bool scales_of_a = w < 2 * WM;
  const int s_wave = scales_of_a ? w : (w - 2 * WM < 4 ? w - 2 * WM : 3);   // which 32 rows of the operand
  {
    int r = (scales_of_a ? m_begin : n_begin) + s_wave * 32 + (lane & 31);
    const int end = scales_of_a ? p.M : p.N;
    r = r < end ? r : end - 1;
    s_off = (unsigned)r * row_scales;
  }
  const uint8_t* ga = p.A + (size_t)s_begin * kRowBytes;
  const uint8_t* gb = p.B + (size_t)s_begin * kRowBytes;
  const uint8_t* gs = (scales_of_a ? p.As : p.Bs) + (size_t)s_begin * kScaleRow;
  const unsigned lds_base = (unsigned)(uintptr_t)lds;
  const unsigned to_a = (unsigned)(WM * w) * 1024, to_b = (unsigned)G::kOffB + (unsigned)w * 2048,
                 to_s = (unsigned)G::kOffS + (unsigned)((scales_of_a ? 0 : G::kRows) + s_wave * 32) * kScaleRow;
  unsigned load_to = lds_base;   // stage buffer that the next load fills
  auto issue = [&](int s) {      // s counts from 0 in the slice; stages are issued in order
    if (tail && s == stages) {
      // move the pieces back to where the row ends.  The offsets are unsigned 32-bit: the bases go back by one stage (there is
      // one) and the offsets forward by it, so that row 0 does not wrap.
      ga -= kRowBytes;
      gb -= kRowBytes;
      gs -= kScaleRow;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        // a whole chunk inside the row, the chunk that is only half inside 8 bytes early, and instead of a chunk behind
        // the row's end the 16 bytes around the tail's start
        auto fix = [&](int c) { return kRowBytes + (2 * c + 2 <= tail_blocks ? 0 : (2 * c < tail_blocks ? -8 : -16 * c - 8)); };
        a_off[i] += (unsigned)fix(chunk_a[i]);
        b_off[i] += (unsigned)fix(chunk_b[i]);
      }
      s_off += (unsigned)tail_blocks;   // one stage forward, 16 - tail_blocks back
    }
    const unsigned to = __builtin_amdgcn_readfirstlane(load_to);
    load_stage<WM>(__builtin_amdgcn_readfirstlane(s < loads ? 1 : 0), to + to_a, to + to_b, to + to_s, ga, gb, gs, a_off, b_off, s_off);
    ga += kRowBytes;
    gb += kRowBytes;
    gs += kScaleRow;
    load_to = load_to + G::kStage == lds_base + G::kLds ? lds_base : load_to + G::kStage;
  };

  // ---- fragments -----------------------------------------------------------------------------------------------------
  const int rho = lane & 31, h = lane >> 5;
  const int row[2] = {wm * 64 + rho, wn * 64 + pi_row(rho)};   // of A and of B, + 32 i
  const unsigned frag[2] = {(unsigned)(row[0] * kRowBytes + ((h ^ ((row[0] >> 1) & 7)) * 16)),
                            (unsigned)(G::kOffB + row[1] * kRowBytes + ((h ^ ((row[1] >> 1) & 7)) * 16))};
  const unsigned srow[2] = {(unsigned)(G::kOffS + row[0] * kScaleRow), (unsigned)(G::kOffS + (G::kRows + row[1]) * kScaleRow)};

  v16f acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = v16f{};
  v4i raw[2][2][2];   // [64-element group, two in flight][operand][32-row block]: 32 codes
  int scw[2][2][2];   // ... the dword with their scale bytes
  v2h sc[2][2][2];    // ... and their two scales
  v8h fr[2][2][2];    // [step, two in flight][operand][block]

  // 64-element group j of this wave in the stage at sb; the wave groups take the stage's four groups in turn
  auto fetch = [&](unsigned sb, int j, int slot) {
    const unsigned u = (unsigned)(kg + j * G::kGroups);
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        raw[slot][o][i] = lds_read16(sb + (frag[o] ^ (u * 32)) + i * 4096);
        scw[slot][o][i] = lds_read4(sb + srow[o] + i * (32 * kScaleRow) + u * 4);
      }
  };
  auto scales = [&](int slot) {   // scale blocks 4 u + 2 h, 4 u + 2 h + 1 of the rows
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int i = 0; i < 2; ++i) sc[slot][o][i] = scale_pair(scw[slot][o][i] >> (16 * h));
  };
  auto convert = [&](int slot, int d, int to) {
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int i = 0; i < 2; ++i) fr[to][o][i] = dequant8((unsigned)raw[slot][o][i][d], sc[slot][o][i][d >> 1]);
  };
  auto multiply = [&](int from) {
#pragma unroll
    for (int nj = 0; nj < 2; ++nj)
#pragma unroll
      for (int mi = 0; mi < 2; ++mi)
        acc[nj][mi] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[from][1][nj], fr[from][0][mi], acc[nj][mi], 0, 0, 0);
  };

  issue(0);
  issue(1);
  issue(2);
  wait_stages<G::kLoads>(__builtin_amdgcn_readfirstlane(loads > 2 ? 2 : loads - 1));
  __syncthreads();
  fetch(lds_base, 0, 0);
  scales(0);
  convert(0, 0, 0);
  unsigned sb = lds_base;
  for (int s = 0; s < stages; ++s) {
    const unsigned sbn = sb + G::kStage == lds_base + G::kLds ? lds_base : sb + G::kStage;
#pragma unroll
    for (int t = 0; t < G::kSteps; ++t) {
      if (t == G::kSteps - 4) {
        // the next stage has landed when only the one behind it is outstanding (the last stages: nothing)
        wait_stages<G::kLoads>(__builtin_amdgcn_readfirstlane(s + 2 < loads ? 1 : 0));
        __syncthreads();   // ... for every wave, and the buffer of the stage before this one is free
        issue(s + 3);
      }
      // a group's fragments are requested two steps before its first conversion, which is a step before its first MFMA (behind
      // the last stage they are what the ring happens to hold, and not used)
      if ((t & 3) == 1) fetch(t + 3 < G::kSteps ? sb : sbn, t + 3 < G::kSteps ? (t + 3) >> 2 : 0, ((t >> 2) + 1) & 1);
      if ((t & 3) == 2) scales(((t >> 2) + 1) & 1);
      convert(((t + 1) >> 2) & 1, (t + 1) & 3, (t + 1) & 1);
      multiply(t & 1);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);   // eight VALU
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (G::kSteps == 4) {   // an odd number of groups per stage: the next stage's group is in the other slot
#pragma unroll
      for (int o = 0; o < 2; ++o)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          raw[0][o][i] = raw[1][o][i];
          sc[0][o][i] = sc[1][o][i];
        }
    }
    sb = sbn;
  }
  if (tail) {   // `sb` is its buffer; it has landed and every wave knows (the last stage's barrier, or the one in front of the loop)
    for (int j = 0; j < 4 / G::kGroups; ++j) {
      const int u = kg + j * G::kGroups;
      if (4 * u >= tail_blocks) break;
      const int b0 = 4 * u + 2 * h;              // this lane's two blocks are b0 and b0 + 1
      const int have = tail_blocks - b0;         // of which the row holds: 2 and more, 1, none
#pragma unroll
      for (int o = 0; o < 2; ++o)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const v4i r = lds_read16(sb + (frag[o] ^ ((unsigned)u * 32)) + i * 4096);
          const v4i half = {r[2], r[3], 0, 0}, none = {0, 0, 0, 0};
          raw[0][o][i] = have >= 2 ? r : (have == 1 ? half : none);
          const unsigned at = sb + srow[o] + i * (32 * kScaleRow) + (unsigned)(16 - tail_blocks) + (unsigned)(have > 0 ? b0 : 0);
          const int first = lds_read1(at), second = lds_read1(have >= 2 ? at + 1 : at);
          sc[0][o][i] = scale_pair((have >= 1 ? first : 0) | (have >= 2 ? second << 8 : 0));
        }
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        convert(0, d, 0);
        multiply(0);
      }
    }
  }

  // ---- the wave groups' sums meet in LDS: of the four 32 x 32 blocks of a part, every group finishes its share ----------
  constexpr int kShare = 4 / G::kGroups;   // blocks that a wave finishes: 2 (both of nj = kg) / 1 (block kg)
  const float g = p.Ag[0] * p.Bg[0];
  __syncthreads();   // the ring is free
  const unsigned part_base = lds_base + (unsigned)(wm * 2 + wn) * (G::kGroups * 4 * 4096u) + (unsigned)lane * 16;   // [group][block][4][64 lanes][16 B]
#pragma unroll
  for (int b = 0; b < 4; ++b)
    if (b / kShare != kg) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const v16f& v = acc[b >> 1][b & 1];
        lds_write16f(part_base + (unsigned)((kg * 4 + b) * 4 + q) * 1024, v4f{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]});
      }
    }
  __syncthreads();
#pragma unroll
  for (int own = 0; own < G::kGroups; ++own)
    if (own == kg) {
#pragma unroll
      for (int b = own * kShare; b < (own + 1) * kShare; ++b) {
        v16f sum = v16f{};
#pragma unroll
        for (int other = 0; other < G::kGroups; ++other) {
          if (other == own) {
            sum += acc[b >> 1][b & 1];
          } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const v4f v = lds_read16f(part_base + (unsigned)((other * 4 + b) * 4 + q) * 1024);
#pragma unroll
              for (int e = 0; e < 4; ++e) sum[4 * q + e] += v[e];
            }
          }
        }
        const v16f out[1][1] = {{sum}};
        const int m0 = m_begin + wm * 64 + 32 * (b & 1), n0 = n_begin + wn * 64 + 32 * (b >> 1);
        if constexpr (SPLITK) store_wave_block_f32<1, 1>(out, p.P + (size_t)slice * (size_t)p.M * (size_t)p.N, p.N, m0, p.M, n0, lane, g);
        else store_wave_block<1, 1>(out, p.C, p.N, m0, p.M, n0, lane, g);
      }
    }
}

template <int WM>
hipError_t launch(const NvArgs& p, bool split, hipStream_t s) {
  using G = Geo<WM>;
  const int m_tiles = (p.M + G::kRows - 1) / G::kRows, n_tiles = (p.N + BN - 1) / BN;
  if (split) {
    if (hipError_t e = allow_dynamic_lds<nv_narrow_kernel<WM, true>>(G::kLds); e != hipSuccess) return e;
    hipLaunchKernelGGL((nv_narrow_kernel<WM, true>), dim3((unsigned)(m_tiles * n_tiles * p.slices)), dim3(kWaves * 64), G::kLds, s, p,
                       m_tiles, n_tiles);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    return launch_splitk_reduce(p.P, p.C, (size_t)p.M * (size_t)p.N, p.slices, s);
  }
  if (hipError_t e = allow_dynamic_lds<nv_narrow_kernel<WM, false>>(G::kLds); e != hipSuccess) return e;
  hipLaunchKernelGGL((nv_narrow_kernel<WM, false>), dim3((unsigned)(m_tiles * n_tiles)), dim3(kWaves * 64), G::kLds, s, p, m_tiles,
                     n_tiles);
  return hipGetLastError();
}

}  // namespace

// Rows in 8-byte steps (K % 16), 32-bit offsets, at least one whole stage.
bool nv_narrow_supports(const NvArgs& p) {
  if (p.M <= 0 || p.N <= 0 || p.K < BK || p.K % 16 != 0) return false;
  // (a tail's offsets lie up to one stage beyond the row's)
  if ((uint64_t)p.M * (uint64_t)(p.K / 2) >= (1ull << 32) - 512 || (uint64_t)p.N * (uint64_t)(p.K / 2) >= (1ull << 32) - 512) return false;
  const uint64_t tiles = (uint64_t)((p.M + 63) / 64) * (uint64_t)((p.N + BN - 1) / BN);
  return tiles < (1ull << 31) && ((reinterpret_cast<uintptr_t>(p.A) | reinterpret_cast<uintptr_t>(p.B)) & 7) == 0;
}

hipError_t launch_nv_narrow(const NvArgs& p, int tile_rows, bool split, hipStream_t s) {
  return tile_rows == 64 ? launch<1>(p, split, s) : launch<2>(p, split, s);
}

// The cheapest kernel by a model of their times on 256 compute units, in microseconds, fitted to graph replays of 60 shapes
// (1 .. 4096 rows, K = 512 .. 15360; within 15 % of nearly all of them):
//  * the weight-streaming kernels (up to 64 rows): 2.5 + K x (what a unit's items cost: a row block 3.6e-4, a tile 3.5e-4 +
//    0.45e-4 per row block), a fifth more where K is no whole number of their panels; register form 6e-4 per item;
//  * 128-column tiles: per round of workgroups 1.04 (64 rows) or 1.62 (128 rows; 1.82 when they fill the chip: the clock gives
//    way) per stage of 256 elements and 4 or 6.5 around them; a split of K adds its partial sums at 7 TB/s there and back,
//    and 3 for the second launch;
//  * 256 x 256 tiles: 5.9 per stage (K % 256 == 0; also in slices), f16-staged 6.9 (K % 64 == 0; other K three times that and never taken).
// Examples, before (256 x 256 tiles, the f16-staged or the one-wave-per-block kernel) and after: 64 x 28672 x 4096 28.7 -> 21.9 us,
// 64 x 5120 x 13824 40.0 -> 19.8, 128 x 28672 x 4096 41.2 -> 34.1, 1024 x 4096 x 4096 62.8 -> 34.9, 451 x 4096 x 4992 114.8 -> 25.8,
// 203 x 3584 x 5760 87.2 -> 22.3, 1272 x 2048 x 11648 272 -> 77, 3066 x 7168 x 3888 443 -> 194, 16 x 4096 x 4176 81.4 -> 11.2.
// K below 1024 that is no multiple of 256 keeps the rules it had (a few microseconds either way).
NvPlan nv_plan(int M, int N, int K, int cus, bool may_split) {
  NvPlan best;
  if (cus <= 0) cus = 256;
  if (M <= 0 || N <= 0 || K < BK || K % 16 != 0 || (K < 4 * BK && K % BK != 0)) return best;
  auto ceil_div = [](long a, long b) { return (a + b - 1) / b; };
  double cost = 1e30;
  auto offer = [&](double c, NvPlan::Kernel k) {
    if (c >= cost) return false;
    cost = c;
    best = NvPlan{};
    best.kernel = k;
    return true;
  };
  const double stages = (double)K / BK;
  const bool ring = K % 32 == 0 && K >= 512 && (M <= 32 || (K / 512) % 2 == 0);
  if (M <= 64 && (ring || K % 128 == 0)) {
    const int mb = M <= 16 ? 1 : (M <= 32 ? 2 : 4), tiles = (int)ceil_div(N, 16);
    const int t = tiles_per_workgroup(tiles, cus, ring || mb == 1 ? 7 : (mb == 2 ? 6 : 4));
    const double per_k = ring ? mb * 3.6e-4 + t * (3.5e-4 + mb * 0.45e-4) : (t + mb) * 6e-4;
    offer(2.5 + ceil_div(ceil_div(tiles, t), cus) * per_k * K * (ring && K % (mb == 4 ? 1024 : 2048) != 0 ? 1.2 : 1.0), NvPlan::kDecode);
  }
  const long tiles256 = ceil_div(M, 256) * ceil_div(N, 256);
  // at least two slices: half of the chip idle with 256 x 256 tiles and a few stages -- callers that provide a
  // workspace have had K split for these shapes (a slice too many costs 1 us at four stages)
  const bool must_split = may_split && M > 64 && K % BK == 0 && K / BK >= 4 && tiles256 * 2 <= cus;
  auto tiled = [&](NvPlan::Kernel kernel, int rows, long tiles, double per_stage, double around, bool splits) {
    if (!must_split || tiles * 2 > cus) {
      if (offer(ceil_div(tiles, cus) * (stages * per_stage + around) + 1.0, kernel)) best.tile_rows = rows;
    }
    if (!splits || !may_split || tiles * 2 > cus) return;
    const int whole = K / BK;
    for (int want = 2; want <= whole && tiles * want <= cus; ++want) {
      const int per = (int)ceil_div(whole, want), slices = (int)ceil_div(whole, per);
      if (slices != want) continue;   // the same slices as a smaller `want`
      const double sums = (double)slices * M * N * sizeof(float);
      if (offer((per + (K % BK) / (double)BK) * per_stage + around + 4.0 + 2.0 * sums / 7e6, kernel)) {
        best.tile_rows = rows;
        best.slices = slices;
        best.slice_stages = per;
        best.workspace_bytes = (size_t)slices * (size_t)M * (size_t)N * sizeof(float);
      }
    }
  };
  const long tiles128 = ceil_div(M, 128) * ceil_div(N, BN);
  tiled(NvPlan::kNarrow, 64, ceil_div(M, 64) * ceil_div(N, BN), 1.04, 4.0, true);
  tiled(NvPlan::kNarrow, 128, tiles128, tiles128 * 5 > 4 * cus ? 1.82 : 1.62, 6.5, true);
  if (K % BK == 0) tiled(NvPlan::kTile, 256, tiles256, 5.9, 4.0, true);
  else if (K % 64 == 0) tiled(NvPlan::kTileF16, 256, tiles256, 6.9, 4.0, false);
  return best;
}

}  // namespace ave
