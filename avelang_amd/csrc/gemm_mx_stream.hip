// MXFP4 GEMM for gfx950 for expert layers with a few rows per expert (a decode batch, or many experts), and for one matrix with few
// weight rows, K whole or in slices: 32, 64 or 128 rows of A by 128 weight rows per tile, and a ring of LDS buffers that never runs
// dry between tiles.
//
// Bound by HBM: every expert's weights are read once, 1.06 bytes per two elements, at 5.2 - 5.7 TB/s over all compute units (21 - 22 KB
// per us each).  The rows of A come from L2 (a stage of 32 KB has been seen to pass in 0.47 us), but a tile of 128 rows brings 112
// repeats of its last row for an expert with 16, and the ring that 128-row tiles started anew for every tile, with a K tail read from global
// memory at its end, ran dry where K is no multiple of 1024.  Here a stage (256 elements of K) is 20, 24 or 32 KB of which 16 are weights;
// six, five or three of them are in flight, and tile boundaries and K tails are ordinary stages of one continuous stream.
//
// Six wavefronts (128 rows: eight): waves 0 and 1 (0 - 3) multiply -- 64 weight rows each, two 32-row blocks, so that with SWIGLU the gate and
// the up value of an output meet in one lane as in gemm_mx_narrow.hip -- and the last four load, a quarter of a stage each, with one
// barrier per stage: behind the barrier of stage j, which says that stage j has landed and stage j - 1 is consumed, stage j + ring - 1
// is requested into the buffer of stage j - 1.  One workgroup per compute unit walks the tiles pid, pid + gridDim.x, ...
//
// Layout, swizzle, K order inside a stage and the epilogues are those of gemm_mx_narrow.hip; the scale rows of one or two
// pairs of stages (16 bytes each) travel with their first stage into slots of their own.  K tail: stages = ceil(K / 256); in the last one 16-byte chunks behind
// the row's end repeat its last chunk, the 16 scale bytes are the row's last 16 (the row may be the tensor's last), and the
// multiplying waves find them there and zero what is not in the row.
#include <cmath>

#include "fp4_common.hpp"
#include "kernels.hpp"
#include "tile_common.hpp"
#include "tile_map.hpp"

namespace ave {
namespace {

constexpr int BN = 128, BK = 256;
constexpr int kRowBytes = BK / 2;   // 128
constexpr int kLoadWaves = 4;

template <int R, bool CHUNKS>   // rows of A per tile; scale rows in chunks of two pairs of stages where LDS has room for them
struct Geo {
  static constexpr int kWM = R == 128 ? 2 : 1;               // multiplying waves along M, R / kWM rows each
  static constexpr int kMI = R / 32 / kWM;                   // 32-row blocks of such a wave
  static constexpr int kMulWaves = 2 * kWM;
  static constexpr int kThreads = (kMulWaves + kLoadWaves) * 64;
  static constexpr int kOffB = R * kRowBytes;
  static constexpr int kStage = kOffB + BN * kRowBytes;      // 20480 / 24576 / 32768
  static constexpr int kRing = R == 32 ? 7 : (R == 64 ? 6 : 4);
  // A chunk's 32 bytes of a row mostly lie in
  // one line, so a load asks for half as many lines as with 16-byte pieces, which were a third of all that the kernel asked for.
  // Slot j of row r holds piece j ^ (r >> 3 & 1): the rows of a read then fall into different banks.  For experts' weights from HBM
  // (scale_chunks, with the figures).  Whole expert layers, pairs -> chunks, us: 300 rows of 8 experts, 4096 / 14336, 187.0 -> 177.4; 1000
  // rows of 128 experts, 2880 / 2880, 359.6 -> 351.4; level at 64 rows of 8 experts.
  static constexpr int kPairs = R == 64 || !CHUNKS ? 1 : 2;
  static constexpr int kScaleRows = R + BN;                  // of a chunk: A's, then B's
  static constexpr int kScaleRow = 16 * kPairs;
  static constexpr int kSlot = kScaleRows * kScaleRow;       // chunks: 5120 / 3072 / 8192
  // Chunks that stages j .. j + kRing - 1 touch at most, a work item having two stages or more: between a chunk's request and
  // that of the one kSlots in front of it lie kSlots - 1 whole chunks, kRing - 1 stages or more (five stages: chunks of
  // four and of one in turn; pairs, three stages: of two and of one).
  static constexpr int kSlots = R == 128 ? 3 : (kPairs == 1 ? 5 : 4);
  static constexpr int kScaleBase = kRing * kStage;
  static constexpr int kLds = kScaleBase + kSlots * kSlot;   // chunks: 163840 / 162816 / 155648
  static constexpr int kALoads = R / 32;                     // 1 KB pieces (8 rows) of A per loading wave and stage
  static constexpr int kData = kALoads + 4;                  // loads of a loading wave for a stage; kPairs more with a chunk's scales
  static constexpr int kWaveRows = kScaleRows / kLoadWaves;  // 40 / 48 / 64 scale rows of a loading wave
  static constexpr int kLoadRows = 64 / kPairs;              // ... of which a load brings this many at most
};
static_assert(Geo<32, true>::kLds <= 160 * 1024 && Geo<64, true>::kLds <= 160 * 1024 && Geo<128, true>::kLds <= 160 * 1024, "LDS of one compute unit");
static_assert(Geo<32, false>::kLds <= 160 * 1024 && Geo<64, false>::kLds <= 160 * 1024 && Geo<128, false>::kLds <= 160 * 1024, "LDS of one compute unit");

__device__ inline int lds_read1(unsigned addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) unsigned char*>((uintptr_t)addr);
}
template <int N>
__device__ inline void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// 16 bytes per lane from an address of its own, lanes below `lanes` only (the instruction counts on vmcnt all the same)
template <int LANES>
__device__ inline void load_scale_rows(const uint8_t* from, unsigned to) {
  unsigned long long saved;
  asm volatile(
      "s_mov_b32 m0, %[to]\n\t"
      "s_mov_b64 %[sv], exec\n\t"
      "s_mov_b64 exec, %[mask]\n\t"
      "global_load_lds_dwordx4 %[from], off\n\t"
      "s_mov_b64 exec, %[sv]\n\t"
      : [sv] "=&s"(saved)
      : [to] "s"(to), [mask] "s"(LANES == 64 ? ~0ull : (1ull << (LANES & 63)) - 1), [from] "v"(from)
      : "m0", "memory");
}

// dma16 for the lanes of `lanes` only (with no lane left it counts on vmcnt all the same)
__device__ inline void dma16_lanes(const void* gbase, unsigned voff, unsigned lds_addr, unsigned long long lanes) {
  unsigned long long saved;
  asm volatile(
      "s_mov_b32 m0, %[to]\n\t"
      "s_mov_b64 %[sv], exec\n\t"
      "s_mov_b64 exec, %[mask]\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %[off], %[base]\n\t"
      "s_mov_b64 exec, %[sv]\n\t"
      : [sv] "=&s"(saved)
      : [to] "s"(__builtin_amdgcn_readfirstlane(lds_addr)), [mask] "s"(lanes), [off] "v"(voff), [base] "s"(gbase)
      : "m0", "memory");
}

// a pointer that is the same in every lane, in scalar registers
__device__ inline const uint8_t* uniform(const uint8_t* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  return reinterpret_cast<const uint8_t*>((uint64_t)hi << 32 | lo);
}

// Experts' first and end rows, clamped to [0, M]: lane l keeps those of experts l, l + 64, l + 128 and l + 192 (none: 0, 0).
constexpr int kSets = 4;
__device__ __forceinline__ void load_table(const MxArgs& p, int (&g_r0)[kSets], int (&g_r1)[kSets]) {
#pragma unroll
  for (int q = 0; q < kSets; ++q) {
    const int e = 64 * q + (int)(threadIdx.x & 63);
    int r0 = 0, r1 = 0;
    if (e < p.E) {
      r0 = p.row_offsets[e];
      r1 = p.row_offsets[e + 1];
      r0 = r0 < 0 ? 0 : (r0 > p.M ? p.M : r0);
      r1 = r1 < 0 ? 0 : (r1 > p.M ? p.M : r1);
    }
    g_r0[q] = r0;
    g_r1[q] = r1;
  }
}
__device__ inline bool table_in_registers(const MxArgs& p) { return p.E <= 64 * kSets; }

// GROUPED: the rows of A belong to p.E experts (p.row_offsets) with weights of their own; otherwise one matrix of p.M rows.
// SPLITK (plain form, not grouped): a work item is a tile and a slice of p.slice_pairs pairs of stages (the last one what is left, the
// K tail with it); its fp32 sums go to p.P[slice][M][N].
// SHIFT: rows that do not all start at a cache line.  A stage cut at the row's start then touches two lines of 128 bytes per row and
// half of what the load path moves is thrown away (5760 x 2880, 16 rows of each of 128 experts: 255 us, with K = 2816 instead 203).
// So a ring buffer holds one LINE per row -- line j of a row that starts 16 sh bytes behind a line boundary is its chunks
// 8 j - sh .. + 7 -- and a stage is read from two buffers: chunk c of stage s lies in line s where c + sh < 8 and in line s + 1
// otherwise (a "late" chunk), in either case in the slot that it has without SHIFT, so that reads stay free of bank conflicts.  Stage s waits for line
// s + 1, one stage earlier than without; a tile whose last stage has late chunks takes one line more.  Chunks of a line that are not the
// row's are not loaded.  Measured: 255 -> 220 us, with 2880 weight rows 131 -> 112.
template <int R, bool SWIGLU, bool QUANT, bool GROUPED, bool SPLITK, bool SHIFT, bool CHUNKS>
__device__ __forceinline__ void stream_tiles(const MxArgs& p, int n_tiles, const int (&g_r0)[kSets], const int (&g_r1)[kSets]) {
  using G = Geo<R, CHUNKS>;
  static_assert(SWIGLU || !QUANT, "the fused quantiser follows the fused SwiGLU");
  static_assert(!SPLITK || (!SWIGLU && !GROUPED), "K is split for the plain GEMM");
  static_assert((!SHIFT && !CHUNKS) || GROUPED, "by lines, scale rows in chunks: the experts' weights only");
  constexpr int kTileN = SWIGLU ? BN / 2 : BN;   // output columns per tile
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const unsigned lds_base = (unsigned)(uintptr_t)lds;
  const unsigned row_bytes = (unsigned)p.K / 2, row_scales = (unsigned)p.K / 32;
  const int stages = (p.K + BK - 1) / BK;
  const int tail_blocks = (p.K % BK) / 32;             // blocks of 32 in the last stage, 0: it is a whole one
  const int pair_tail = (p.K % (2 * BK)) / 32;         // scale bytes in the last pair, 0: all 16
  // SHIFT: rows start at multiples of `unit` chunks behind a line boundary; row r of a matrix at chunk (base + r * row16) % 8
  const unsigned row16 = row_bytes / 16, a16 = (unsigned)(reinterpret_cast<uintptr_t>(p.A) >> 4), b16 = (unsigned)(reinterpret_cast<uintptr_t>(p.B) >> 4);
  const unsigned bits16 = row16 | a16 | b16 | 8;
  const int unit = (int)(bits16 & (0u - bits16));
  const bool late_at_end = SHIFT && (tail_blocks != 0 ? tail_blocks : 8) > unit;   // the last stage of K has late chunks in some row

  // Beside its experts' rows a lane keeps their {first m-tile, m-tiles}; with more than 256 experts the caller's table is walked for
  // every tile.
  int g_first[kSets], g_nt[kSets];
  int m_tiles = 0;
  const bool in_registers = table_in_registers(p);
  if (!GROUPED) {
    m_tiles = (p.M + R - 1) / R;
  } else if (in_registers) {
#pragma unroll
    for (int q = 0; q < kSets; ++q) {
      const int nt = g_r1[q] > g_r0[q] ? (g_r1[q] - g_r0[q] + R - 1) / R : 0;
      int incl = nt;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int up = __shfl_up(incl, d);
        if (lane >= d) incl += up;
      }
      g_first[q] = m_tiles + incl - nt;
      g_nt[q] = nt;
      m_tiles += __builtin_amdgcn_readlane(incl, 63);
    }
  } else {
    m_tiles = (p.M + R - 1) / R + p.E;   // upper bound
  }
  const int total = m_tiles * n_tiles * (SPLITK ? p.slices : 1);

  int pid = (int)blockIdx.x - (int)gridDim.x;
  int m_begin = 0, m_end = 0, expert = 0, n_begin = 0;
  int slice = 0, s_first = 0, s_last = stages;   // stages of the tile: all of them, or those of a slice
  auto next_tile = [&]() {   // false: no tile left; uniform for the workgroup
    while ((pid += (int)gridDim.x) < total) {
      int tm, tn, id = pid;
      if (SPLITK) {
        slice = id / (m_tiles * n_tiles);
        id -= slice * (m_tiles * n_tiles);
        s_first = slice * 2 * p.slice_pairs;
        s_last = s_first + 2 * p.slice_pairs < stages && slice + 1 < p.slices ? s_first + 2 * p.slice_pairs : stages;
      }
      map_tile(id, m_tiles, n_tiles, tm, tn);
      n_begin = tn * kTileN;
      if (!GROUPED) {
        m_begin = tm * R;
        m_end = p.M;
        return true;
      }
      if (!in_registers) {
        int e, r0, r1;
        if (!__builtin_amdgcn_readfirstlane(locate_group_tile(p.row_offsets, p.E, p.M, R, tm, e, r0, r1) ? 1 : 0)) continue;
        expert = __builtin_amdgcn_readfirstlane(e);
        m_begin = __builtin_amdgcn_readfirstlane(r0);
        m_end = __builtin_amdgcn_readfirstlane(r1);
        return true;
      }
#pragma unroll
      for (int q = 0; q < kSets; ++q) {
        const unsigned long long hits = __ballot(tm >= g_first[q] && tm < g_first[q] + g_nt[q]);
        if (hits) {
          const int e = __builtin_ctzll(hits);
          expert = 64 * q + e;
          m_begin = __builtin_amdgcn_readlane(g_r0[q], e) + (tm - __builtin_amdgcn_readlane(g_first[q], e)) * R;
          m_end = __builtin_amdgcn_readlane(g_r1[q], e);
          return true;
        }
      }
    }
    return false;
  };
  // row of B behind row `row` (0 .. 127) of the tile's B image, clamped to a valid row
  auto b_image_row = [&](int row) {
    if (SWIGLU) {   // rows 64 w + j: j < 32 the gate row, j >= 32 the up row of output column 32 w + (j & 31)
      int n = n_begin + 32 * (row >> 6) + (row & 31);
      n = n < p.N ? n : p.N - 1;
      return (row & 32) ? p.N + n : n;
    }
    const int n = n_begin + row;
    return n < p.N ? n : p.N - 1;
  };

  if (w >= G::kMulWaves) {
    // ---- loading waves ---------------------------------------------------------------------------------------------------
    const int wi = w - G::kMulWaves;
    unsigned a_off[G::kALoads], b_off[4];
    int a_chunk[G::kALoads], b_chunk[4];
    unsigned a_late = 0, b_late = 0;   // SHIFT: bit i: this lane's chunk of load i is a late one
    const uint8_t *ga = nullptr, *gb = nullptr, *gs = nullptr;
    [[maybe_unused]] const uint8_t* gs_up = nullptr;   // chunks: rows 32 .. of the wave's, and the piece of a row that this lane fetches
    [[maybe_unused]] int s_from = 0;
    int s = 0, s_end = 0;      // stage (SHIFT: line) of the tile that goes out next, and the one behind its last
    unsigned to = lds_base, slot_to = lds_base + G::kScaleBase;
    unsigned with_scales = 0;  // bit i: the stage issued i stages ago brought scale rows
    int issued = 0;
    auto issue = [&]() {       // false: nothing left
      if (s == s_end) {
        if (!next_tile()) return false;
        s = s_first;
        s_end = s_last + (late_at_end ? 1 : 0);
        a_late = b_late = 0;
        const int lr = lane >> 3, cprime = lane & 7;
#pragma unroll
        for (int i = 0; i < G::kALoads; ++i) {
          const int row = (wi * G::kALoads + i) * 8 + lr;
          int am = m_begin + row;
          am = am < m_end ? am : m_end - 1;
          a_chunk[i] = cprime ^ ((row >> 1) & 7);
          a_off[i] = (unsigned)am * row_bytes + (unsigned)a_chunk[i] * 16;
          if (SHIFT) {
            if (a_chunk[i] + (int)((a16 + (unsigned)am * row16) & 7) >= 8) a_late |= 1u << i;
            else a_off[i] += kRowBytes;
          }
        }
        const size_t expert_rows = (size_t)expert * (SWIGLU ? 2 : 1) * p.N;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = (wi * 4 + i) * 8 + lr;
          b_chunk[i] = cprime ^ ((row >> 1) & 7);
          const unsigned bn = (unsigned)b_image_row(row);
          b_off[i] = bn * row_bytes + (unsigned)b_chunk[i] * 16;
          if (SHIFT) {
            if (b_chunk[i] + (int)((b16 + ((unsigned)expert_rows + bn) * row16) & 7) >= 8) b_late |= 1u << i;
            else b_off[i] += kRowBytes;
          }
        }
        // (SHIFT: a late chunk is that of the stage before; the offsets are from one stage in front of line s)
        ga = p.A + (size_t)s * kRowBytes - (SHIFT ? kRowBytes : 0);
        gb = p.B + expert_rows * row_bytes + (size_t)s * kRowBytes - (SHIFT ? kRowBytes : 0);
        if constexpr (G::kPairs == 1) {
          const int sr = wi * G::kWaveRows + (lane < G::kWaveRows ? lane : 0);
          int am = m_begin + sr;
          am = am < m_end ? am : m_end - 1;
          gs = sr < R ? p.As + (size_t)am * row_scales : p.Bs + (expert_rows + (unsigned)b_image_row(sr - R)) * row_scales;
          gs += (size_t)(s >> 1) * 16;
        } else {
          auto scale_row = [&](int in_wave) {
            const int sr = wi * G::kWaveRows + (in_wave < G::kWaveRows ? in_wave : 0);
            int am = m_begin + sr;
            am = am < m_end ? am : m_end - 1;
            return sr < R ? p.As + (size_t)am * row_scales : p.Bs + (expert_rows + (unsigned)b_image_row(sr - R)) * row_scales;
          };
          gs = scale_row(lane >> 1);
          gs_up = scale_row(G::kLoadRows + (lane >> 1));
          // (kLoadRows is 32 and kWaveRows a multiple of 8: the same piece in both loads)
          s_from = (lane & 1) ^ ((wi * G::kWaveRows + (lane >> 1)) >> 3 & 1);
        }
      }
      if (!SHIFT && tail_blocks != 0 && s == stages - 1) {   // chunks behind the row's end: its last chunk again
#pragma unroll
        for (int i = 0; i < G::kALoads; ++i)
          if (a_chunk[i] >= tail_blocks) a_off[i] -= (unsigned)(a_chunk[i] - (tail_blocks - 1)) * 16;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (b_chunk[i] >= tail_blocks) b_off[i] -= (unsigned)(b_chunk[i] - (tail_blocks - 1)) * 16;
      }
      const bool scales = (G::kPairs == 1 ? (s & 1) == 0 : ((s - s_first) & 3) == 0) && (!SHIFT || s < s_last);
      if (scales) {
        if constexpr (G::kPairs == 1) {
          if (pair_tail != 0 && s + 2 >= stages) gs -= 16 - pair_tail;   // (K >= 512: there are 16 bytes in front of the row's end)
          load_scale_rows<G::kWaveRows>(gs, __builtin_amdgcn_readfirstlane(slot_to) + (unsigned)wi * (G::kWaveRows * 16));
          gs += 16;
        } else {
          const unsigned first = __builtin_amdgcn_readfirstlane(slot_to) + (unsigned)wi * (G::kWaveRows * 32);
          // the last pair's piece, and those behind it, are the row's last 16 bytes
          unsigned at = (unsigned)((s >> 1) + s_from) * 16;
          at = at < row_scales - 16 ? at : row_scales - 16;
          load_scale_rows<64>(gs + at, first);
          load_scale_rows<2 * (G::kWaveRows - G::kLoadRows)>(gs_up + at, first + 1024);
        }
        slot_to = slot_to + G::kSlot == lds_base + G::kLds ? lds_base + G::kScaleBase : slot_to + G::kSlot;
      }
      with_scales = (with_scales << 1) | (scales ? 1u : 0u);
      if (SHIFT && (s == 0 || s >= stages - 1)) {   // a line with chunks that are not the row's: these lanes stay out
        auto mine = [&](unsigned late, int i, int chunk) {
          const int at = 8 * s + chunk - (late >> i & 1 ? 8 : 0);
          return __ballot(at >= 0 && at < (int)row_scales);
        };
#pragma unroll
        for (int i = 0; i < G::kALoads; ++i) dma16_lanes(uniform(ga), a_off[i], to + (unsigned)(wi * G::kALoads + i) * 1024, mine(a_late, i, a_chunk[i]));
#pragma unroll
        for (int i = 0; i < 4; ++i) dma16_lanes(uniform(gb), b_off[i], to + G::kOffB + (unsigned)(wi * 4 + i) * 1024, mine(b_late, i, b_chunk[i]));
      } else {
#pragma unroll
        for (int i = 0; i < G::kALoads; ++i) dma16(uniform(ga), a_off[i], to + (unsigned)(wi * G::kALoads + i) * 1024);
#pragma unroll
        for (int i = 0; i < 4; ++i) dma16(uniform(gb), b_off[i], to + G::kOffB + (unsigned)(wi * 4 + i) * 1024);
      }
      ga += kRowBytes;
      gb += kRowBytes;
      to = to + G::kStage == lds_base + G::kScaleBase ? lds_base : to + G::kStage;
      ++s;
      ++issued;
      return true;
    };
    bool more = true;
    for (int i = 0; i < G::kRing - 1 && more; ++i) more = issue();
    for (int j = 0; j < issued; ++j) {
      // Stage j (SHIFT: line j + 1) has landed when only the loads of the stages behind it are outstanding: `ahead` of them, each kData
      // loads and kPairs more for those that brought scale rows (fewer than there are is safe, and waits a little longer).
      constexpr int kAhead = G::kRing - 2 - (SHIFT ? 1 : 0);   // (while there is more to issue)
      const int ahead = __builtin_amdgcn_readfirstlane(issued - 1 - (SHIFT ? 1 : 0) - j);
      if (ahead >= kAhead) {
        const int c = __popc(__builtin_amdgcn_readfirstlane((int)(with_scales & ((1u << kAhead) - 1))));
        if (c >= 3) wait_vm<kAhead * G::kData + 3 * G::kPairs>();
        else if (c == 2) wait_vm<kAhead * G::kData + 2 * G::kPairs>();
        else if ((G::kPairs == 1 && !SHIFT) || c == 1) wait_vm<kAhead * G::kData + G::kPairs>();   // (pairs, not SHIFT: every two stages in a row hold the first stage of a pair)
        else wait_vm<kAhead * G::kData>();
      } else if (ahead == 4) {
        wait_vm<4 * G::kData>();
      } else if (ahead == 3) {
        wait_vm<3 * G::kData>();
      } else if (ahead == 2) {
        wait_vm<2 * G::kData>();
      } else if (ahead == 1) {
        wait_vm<G::kData>();
      } else {
        wait_vm<0>();
      }
      __syncthreads();
      if (more) more = issue();
    }
    return;
  }

  // ---- multiplying waves ----------------------------------------------------------------------------------------------------
  constexpr int MI = G::kMI;
  const int rho = lane & 31, h = lane >> 5;
  const int wn = w & 1, m_wave = (w >> 1) * (32 * MI);   // this wave's weight rows start at 64 wn, its rows of A at m_wave
  const int a_row = m_wave + rho;             // + 32 mi
  const int b_row = wn * 64 + pi_row(rho);    // + 32 nj
  const unsigned a_frag = (unsigned)(a_row * kRowBytes + (((4 * h) ^ ((a_row >> 1) & 7)) * 16));
  const unsigned b_frag = (unsigned)(G::kOffB + b_row * kRowBytes + (((4 * h) ^ ((b_row >> 1) & 7)) * 16));
  // a row's piece 0 in a slot, + kScaleRow * 32 per 32 rows; piece 1 at the address with bit 4 the other way
  const unsigned a_sc = (unsigned)(a_row * G::kScaleRow + (G::kPairs == 2 ? (a_row >> 3 & 1) * 16 : 0));
  const unsigned b_sc = (unsigned)((R + b_row) * G::kScaleRow + (G::kPairs == 2 ? (b_row >> 3 & 1) * 16 : 0));
  unsigned sb = lds_base, slot = lds_base + G::kLds - G::kSlot;
  auto next_buffer = [&]() { sb = sb + G::kStage == lds_base + G::kScaleBase ? lds_base : sb + G::kStage; };
  while (next_tile()) {
    // SHIFT: bit c: chunk c of the fragment row is a late one
    unsigned a_late[MI] = {}, b_late[2] = {};
    if (SHIFT) {
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        int am = m_begin + a_row + 32 * i;
        am = am < m_end ? am : m_end - 1;
        a_late[i] = 0xFF00u >> ((a16 + (unsigned)am * row16) & 7);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
        b_late[i] = 0xFF00u >> ((b16 + ((unsigned)expert * (SWIGLU ? 2 : 1) * (unsigned)p.N + (unsigned)b_image_row(b_row + 32 * i)) * row16) & 7);
    }
    // where a fragment row's chunk `chunk` lies, from the buffer of its stage
    auto late = [&](unsigned mask, int chunk) {
      if (!SHIFT) return 0u;
      const unsigned to_next = sb + G::kStage == lds_base + G::kScaleBase ? lds_base - sb : (unsigned)G::kStage;
      return (0u - (mask >> chunk & 1)) & to_next;
    };
    v16f acc[2][MI];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < MI; ++j) acc[i][j] = v16f{};
    int as_cur[MI], bs_cur[2];
    // The dword of a row's 16 scale bytes for stage parity P and this lane's half: 2 P + h; chunks: of the piece `piece` bytes into the
    // slot.  (What differs between pairs and chunks is spelled out where it stands, with nothing of the chunks left in the pair forms:
    // one expression for both made the compiler order the pair forms' address arithmetic differently, 1 - 4 % slower on 64- and
    // 128-row tiles: gate+up with quantiser 70 x 2560 x 1792 7.72 -> 7.98 us, plain 100 x 4096 x 2048 7.97 -> 8.15.)
    auto read_scales = [&](int P, [[maybe_unused]] unsigned piece) {
      if constexpr (G::kPairs == 1) {
#pragma unroll
        for (int i = 0; i < MI; ++i) as_cur[i] = lds_read4(slot + a_sc + i * 512 + (unsigned)(2 * P + h) * 4);
#pragma unroll
        for (int i = 0; i < 2; ++i) bs_cur[i] = lds_read4(slot + b_sc + i * 512 + (unsigned)(2 * P + h) * 4);
      } else {
        const unsigned at = slot + (unsigned)(2 * P + h) * 4, as = a_sc ^ piece, bs = b_sc ^ piece;
#pragma unroll
        for (int i = 0; i < MI; ++i) as_cur[i] = lds_read4(at + as + i * 1024);
#pragma unroll
        for (int i = 0; i < 2; ++i) bs_cur[i] = lds_read4(at + bs + i * 1024);
      }
    };
    v4i af[4][MI], bf[4][2];   // the fragments of a whole stage: all requested before the first is waited for
    auto read_frags = [&]() {
#pragma unroll
      for (int kj = 0; kj < 4; ++kj) {
#pragma unroll
        for (int i = 0; i < MI; ++i) af[kj][i] = lds_read16(sb + late(a_late[i], 4 * h + kj) + (a_frag ^ ((unsigned)kj * 16)) + i * 4096);
#pragma unroll
        for (int i = 0; i < 2; ++i) bf[kj][i] = lds_read16(sb + late(b_late[i], 4 * h + kj) + (b_frag ^ ((unsigned)kj * 16)) + i * 4096);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    // stages of whole pairs end here
    const int whole = pair_tail == 0 || s_last < stages ? s_last : (stages - 1) & ~1;
    auto next_slot = [&]() { slot = slot + G::kSlot == lds_base + G::kLds ? lds_base + G::kScaleBase : slot + G::kSlot; };
    int s = s_first;
    auto behind_the_last_stage = [&]() {
      if (late_at_end) {
        __syncthreads();
        next_buffer();
      }
    };
    if (G::kWM > 1 && m_begin + m_wave >= m_end) {   // no rows for this wave: the barriers and the positions, nothing else
      for (; s < s_last; ++s) {
        __syncthreads();
        if (G::kPairs == 1 ? (s & 1) == 0 : ((s - s_first) & 3) == 0) next_slot();
        next_buffer();
      }
      behind_the_last_stage();
      continue;
    }
    for (; s < whole; ++s) {
      __syncthreads();   // the stage has landed
      if (G::kPairs == 1 ? (s & 1) == 0 : ((s - s_first) & 3) == 0) next_slot();
      read_scales(s & 1, G::kPairs == 1 ? 0u : (unsigned)((s - s_first) & 2) * 8);
      read_frags();
#pragma unroll
      for (int nj = 0; nj < 2; ++nj)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) acc[nj][mi] = mfma32<0, 0>(bf[0][nj], af[0][mi], acc[nj][mi], bs_cur[nj], as_cur[mi]);
#pragma unroll
      for (int nj = 0; nj < 2; ++nj)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) acc[nj][mi] = mfma32<1, 1>(bf[1][nj], af[1][mi], acc[nj][mi], bs_cur[nj], as_cur[mi]);
#pragma unroll
      for (int nj = 0; nj < 2; ++nj)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) acc[nj][mi] = mfma32<2, 2>(bf[2][nj], af[2][mi], acc[nj][mi], bs_cur[nj], as_cur[mi]);
#pragma unroll
      for (int nj = 0; nj < 2; ++nj)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) acc[nj][mi] = mfma32<3, 3>(bf[3][nj], af[3][mi], acc[nj][mi], bs_cur[nj], as_cur[mi]);
      next_buffer();
    }
    // The one or two stages behind the last whole pair.  Their blocks are added up in the order of the kernel that runs the
    // ungrouped GEMM of these rows: two by two (gemm_mx_narrow.hip), or four apart as in every other stage (gemm_mx_tile.hip).
    // A block that is not there is zeros under the scale 2^0.
    for (; s < s_last; ++s) {
      __syncthreads();
      if (G::kPairs == 1 ? (s & 1) == 0 : ((s - s_first) & 3) == 0) next_slot();
      const int blocks = s == stages - 1 && tail_blocks != 0 ? tail_blocks : 8;
      if constexpr (GROUPED) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int block = p.tail_four_apart ? 4 * h + j : 2 * j + h;
          const bool have = block < blocks;
          const unsigned at = slot + (unsigned)(16 - pair_tail + 8 * (s & 1) + (have ? block : 0));
          const v4i none = {0, 0, 0, 0};
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            const v4i f = lds_read16(sb + late(a_late[i], block) + (unsigned)((a_row + 32 * i) * kRowBytes + ((block ^ ((a_row >> 1) & 7)) * 16)));
            const int sc = lds_read1(at + (G::kPairs == 1 ? a_sc : a_sc ^ ((unsigned)((s - s_first) & 2) * 8)) + i * (32 * G::kScaleRow));
            af[j][i] = have ? f : none;
            as_cur[i] = have ? sc : 0x7f;
          }
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const v4i f = lds_read16(sb + late(b_late[i], block) + (unsigned)(G::kOffB + (b_row + 32 * i) * kRowBytes + ((block ^ ((b_row >> 1) & 7)) * 16)));
            const int sc = lds_read1(at + (G::kPairs == 1 ? b_sc : b_sc ^ ((unsigned)((s - s_first) & 2) * 8)) + i * (32 * G::kScaleRow));
            bf[j][i] = have ? f : none;
            bs_cur[i] = have ? sc : 0x7f;
          }
#pragma unroll
          for (int nj = 0; nj < 2; ++nj)
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) acc[nj][mi] = mfma32<0, 0>(bf[j][nj], af[j][mi], acc[nj][mi], bs_cur[nj], as_cur[mi]);
        }
      } else {
        // One matrix: all of the stage's fragments and scales are requested before the first is waited for, as in the stages above.
        // Left to the compiler, the plain form's 64-row tiles and all 128-row tiles waited for them one by one: 250 x 1280 x 1376 8.07 ->
        // 7.45 us, 220 x 1536 x 4480 13.7 -> 13.1, 100 x 2048 x 2944 10.8 -> 10.1.  (Grouped, this order was 4 % slower in places, 5 %
        // faster in others.)
        int as_tail[4][MI], bs_tail[4][2];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int block = p.tail_four_apart ? 4 * h + j : 2 * j + h;
          const unsigned at = slot + (unsigned)(16 - pair_tail + 8 * (s & 1) + (block < blocks ? block : 0));
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            af[j][i] = lds_read16(sb + (unsigned)((a_row + 32 * i) * kRowBytes + ((block ^ ((a_row >> 1) & 7)) * 16)));
            as_tail[j][i] = lds_read1(at + a_sc + i * 512);
          }
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            bf[j][i] = lds_read16(sb + (unsigned)(G::kOffB + (b_row + 32 * i) * kRowBytes + ((block ^ ((b_row >> 1) & 7)) * 16)));
            bs_tail[j][i] = lds_read1(at + b_sc + i * 512);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const bool have = (p.tail_four_apart ? 4 * h + j : 2 * j + h) < blocks;
          const v4i none = {0, 0, 0, 0};
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            af[j][i] = have ? af[j][i] : none;
            as_cur[i] = have ? as_tail[j][i] : 0x7f;
          }
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            bf[j][i] = have ? bf[j][i] : none;
            bs_cur[i] = have ? bs_tail[j][i] : 0x7f;
          }
#pragma unroll
          for (int nj = 0; nj < 2; ++nj)
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) acc[nj][mi] = mfma32<0, 0>(bf[j][nj], af[j][mi], acc[nj][mi], bs_cur[nj], as_cur[mi]);
        }
      }
      next_buffer();
    }
    behind_the_last_stage();

    if constexpr (SWIGLU) {
      // acc[0][mi] holds the gate and acc[1][mi] the up values of row m_begin + m_wave + 32 mi + c, outputs n_begin + 32 wn + 16 piece + 8 q
      // + 0..7 (registers 8 piece .. 8 piece + 7)
      const int c = lane & 31, q = lane >> 5;
      const bool vec_ok = (p.N % 8 == 0) && ((reinterpret_cast<uintptr_t>(p.C) & 15) == 0);
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        const int m = m_begin + m_wave + 32 * mi + c;
        if (m >= m_end) continue;
        uint16_t* crow = QUANT ? nullptr : p.C + (size_t)m * p.N;
        v4i o[2];
#pragma unroll
        for (int piece = 0; piece < 2; ++piece) {
          float hv[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) hv[e] = silu(acc[0][mi][8 * piece + e]) * acc[1][mi][8 * piece + e];
          o[piece] = v4i{(int)pack_bf16x2(hv[0], hv[1]), (int)pack_bf16x2(hv[2], hv[3]), (int)pack_bf16x2(hv[4], hv[5]), (int)pack_bf16x2(hv[6], hv[7])};
          if constexpr (!QUANT) {
            const int n = n_begin + 32 * wn + 16 * piece + 8 * q;
            if (vec_ok && n + 8 <= p.N) {
              *reinterpret_cast<v4i*>(crow + n) = o[piece];
            } else {
#pragma unroll
              for (int e = 0; e < 8; ++e)
                if (n + e < p.N) crow[n + e] = (uint16_t)(((unsigned)o[piece][e >> 1] >> (16 * (e & 1))) & 0xFFFF);
            }
          }
        }
        if constexpr (QUANT) {
          // the stand-alone quantiser's steps on the bf16 values (N % 32 == 0: a block lies inside the matrix or outside it as
          // a whole, so both lanes of the exchange are in the same state)
          float v[2][8];
#pragma unroll
          for (int piece = 0; piece < 2; ++piece)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              v[piece][2 * j] = __builtin_bit_cast(float, (unsigned)o[piece][j] << 16);
              v[piece][2 * j + 1] = __builtin_bit_cast(float, (unsigned)o[piece][j] & 0xFFFF0000u);
            }
          unsigned amax = abs_max_bits(v[0]);
          const unsigned second = abs_max_bits(v[1]);
          amax = lane_xor_max_bits(amax > second ? amax : second, 32);
          const int byte = mx_scale_byte(amax);
          const float scale = mx_scale_value(byte);
          const int n0 = n_begin + 32 * wn;   // first output of the block
          if (n0 < p.N) {
#pragma unroll
            for (int piece = 0; piece < 2; ++piece) {
              unsigned codes = 0;
              codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, v[piece][0], v[piece][1], scale, 0);
              codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, v[piece][2], v[piece][3], scale, 1);
              codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, v[piece][4], v[piece][5], scale, 2);
              codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, v[piece][6], v[piece][7], scale, 3);
              *reinterpret_cast<unsigned*>(p.Q + (size_t)m * (q_row_cols(p) / 2) + (n0 + 16 * piece + 8 * q) / 2) = byte == 0xFF ? 0u : codes;
            }
            if (q == 0) p.Qs[(size_t)m * (q_row_cols(p) / 32) + n0 / 32] = (uint8_t)byte;
          }
        }
      }
    } else if constexpr (SPLITK) {
      store_wave_block_f32<MI, 2>(acc, p.P + (size_t)slice * (size_t)p.M * (size_t)p.N, p.N, m_begin + m_wave, m_end, n_begin + wn * 64, lane);
    } else {
      store_wave_block<MI, 2>(acc, p.C, p.N, m_begin + m_wave, m_end, n_begin + wn * 64, lane, 1.0f);
    }
  }
}

template <int R, bool SWIGLU, bool QUANT, bool GROUPED, bool SPLITK, bool SHIFT, bool CHUNKS>
__global__ __launch_bounds__((Geo<R, CHUNKS>::kThreads)) void mx_stream_kernel(MxArgs p, int n_tiles) {
  int g_r0[kSets], g_r1[kSets];
  if (GROUPED && table_in_registers(p)) load_table(p, g_r0, g_r1);
  stream_tiles<R, SWIGLU, QUANT, GROUPED, SPLITK, SHIFT, CHUNKS>(p, n_tiles, g_r0, g_r1);
}

// Rows per tile for the experts' table as it is, from the `rows` that the host took for the average: an expert with more rows than a
// tile sends its weights through the load path once per tile, so where routing is uneven tall tiles take fewer rounds.  The
// cheapest by rounds of the grid x rows that a stage loads, the same in every wave; nothing to look for (and no time spent) where no
// expert has more than one tile.
__device__ __forceinline__ int rows_for_table(const int (&g_r0)[kSets], const int (&g_r1)[kSets], int n_tiles, int rows) {
  int tiles32 = 0, tiles64 = 0, tiles128 = 0, most = 0;
#pragma unroll
  for (int q = 0; q < kSets; ++q) {
    const int n = g_r1[q] > g_r0[q] ? g_r1[q] - g_r0[q] : 0;
    most = n > most ? n : most;
    tiles32 += (n + 31) >> 5;
    tiles64 += (n + 63) >> 6;
    tiles128 += (n + 127) >> 7;
  }
  if (!__any(most > rows)) return rows;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    tiles32 += __shfl_xor(tiles32, d);
    tiles64 += __shfl_xor(tiles64, d);
    tiles128 += __shfl_xor(tiles128, d);
  }
  auto cost = [&](int tiles, int of) { return ceilf((float)tiles * (float)n_tiles / (float)gridDim.x) * (float)(of + BN); };
  const float at64 = cost(tiles64, 64);
  const bool tall = rows == 64 || at64 < cost(tiles32, 32);
  const float least = tall ? at64 : cost(tiles32, 32);
  const int taken = cost(tiles128, 128) < least ? 128 : (tall ? 64 : 32);
  return __builtin_amdgcn_readfirstlane(taken);
}

// Expert layers on tiles of 32 or 64 rows, or (`by_table`) of more where the experts' table asks for it.  Waves that the tile
// height has no work for end at once (a barrier waits for the others alone).  Measured, tiles by the average alone -> by the table
// (128-row tiles with a ring per tile before that), plain, us: 128 rows of 8 experts, 28672 x 4096, all in one expert 31.8 -> 20.0 (21.0);
// 4096 x 14336, routed by 1 / rank 61.2 -> 42.0 (49.1); 2000 rows of 128 experts, 5760 x 2880, on a quarter of them 95.9 -> 78.7 (105), in
// one 80.2 -> 36.7 (46.4), evenly 227.3 and 227.0 (327).
template <bool CHUNKS>
constexpr int kTallestLds = CHUNKS ? Geo<32, true>::kLds : Geo<64, false>::kLds;
template <int R>
constexpr bool fits_taller = Geo<R, true>::kThreads <= Geo<128, true>::kThreads && Geo<R, true>::kLds <= kTallestLds<true> && Geo<R, false>::kLds <= kTallestLds<false>;
static_assert(fits_taller<32> && fits_taller<64> && fits_taller<128>);
template <bool SWIGLU, bool QUANT, bool SHIFT, bool CHUNKS>
__global__ __launch_bounds__((Geo<128, true>::kThreads)) void mx_stream_by_table_kernel(MxArgs p, int n_tiles, int rows, int by_table) {
  int g_r0[kSets], g_r1[kSets];
  if (table_in_registers(p)) {
    load_table(p, g_r0, g_r1);
    if (by_table) rows = rows_for_table(g_r0, g_r1, n_tiles, rows);
  }
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  if (rows == 128) {
    stream_tiles<128, SWIGLU, QUANT, true, false, SHIFT, CHUNKS>(p, n_tiles, g_r0, g_r1);
  } else if (rows == 64) {
    if (wave < Geo<64, true>::kThreads / 64) stream_tiles<64, SWIGLU, QUANT, true, false, SHIFT, CHUNKS>(p, n_tiles, g_r0, g_r1);
  } else {
    if (wave < Geo<32, true>::kThreads / 64) stream_tiles<32, SWIGLU, QUANT, true, false, SHIFT, CHUNKS>(p, n_tiles, g_r0, g_r1);
  }
}

// workgroups for m-tiles of R rows (grouped: an upper bound of the experts' tile lists), at most one per compute unit; 0: no device
template <bool SWIGLU, bool GROUPED, bool SPLITK>
unsigned stream_grid(const MxArgs& p, int rows, int* n_tiles) {
  constexpr int kTileN = SWIGLU ? BN / 2 : BN;
  *n_tiles = (p.N + kTileN - 1) / kTileN;
  const int cus = compute_units();
  const long tiles = ((long)(p.M + rows - 1) / rows + (GROUPED ? p.E : 0)) * *n_tiles * (SPLITK ? p.slices : 1);
  return cus <= 0 ? 0 : (unsigned)(tiles < cus ? tiles : cus);
}
template <int R, bool SWIGLU, bool QUANT, bool GROUPED, bool SPLITK, bool SHIFT, bool CHUNKS>
hipError_t launch(const MxArgs& p, hipStream_t s) {
  int n_tiles;
  const unsigned grid = stream_grid<SWIGLU, GROUPED, SPLITK>(p, R, &n_tiles);
  if (grid == 0) return hipErrorInvalidDevice;
  constexpr auto kernel = mx_stream_kernel<R, SWIGLU, QUANT, GROUPED, SPLITK, SHIFT, CHUNKS>;
  using G = Geo<R, CHUNKS>;
  if (hipError_t e = allow_dynamic_lds<kernel>(G::kLds); e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(G::kThreads), G::kLds, s, p, n_tiles);
  return hipGetLastError();
}
template <bool SWIGLU, bool QUANT, bool SHIFT, bool CHUNKS>
hipError_t launch_grouped_lines(const MxArgs& p, int rows, hipStream_t s) {
  if (rows == 128) return launch<128, SWIGLU, QUANT, true, false, SHIFT, CHUNKS>(p, s);
  int n_tiles;
  const unsigned grid = stream_grid<SWIGLU, true, false>(p, rows, &n_tiles);
  if (grid == 0) return hipErrorInvalidDevice;
  constexpr auto kernel = mx_stream_by_table_kernel<SWIGLU, QUANT, SHIFT, CHUNKS>;
  if (hipError_t e = allow_dynamic_lds<kernel>(kTallestLds<CHUNKS>); e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3((Geo<128, true>::kThreads)), kTallestLds<CHUNKS>, s, p, n_tiles, rows, p.rows_by_table);
  return hipGetLastError();
}
// SHIFT for experts' weights whose rows do not all start at a cache line, from HBM and over a few lines: the start of a tile costs it
// more, and where a launch is short or its weights are in the last-level cache the lines that it saves do not bound it.  Measured on
// weights beyond that cache (200 experts x 8 and x 40 rows, 4096 weight rows; 78 x 4, 21504; 120 x 100, 8192), without against with: K = 544 and 800 0.83 - 1.06,
// 1056 1.03 - 1.13, 1120 and 1184 (five stages and a line more) 0.94 - 1.08, 1312 - 1696 1.02 - 1.18, 2080 - 4256 1.10 - 1.21.  One
// matrix (1 - 300 rows): 0.87 - 1.04, so not there.
template <bool SWIGLU>
bool by_lines(const MxArgs& p) {
  if (p.K <= 4 * BK && !p.by_lines) return false;
  const uint64_t row = (uint64_t)p.K / 2, b_rows = (uint64_t)p.N * (SWIGLU ? 2 : 1);
  const uint64_t at = (reinterpret_cast<uintptr_t>(p.A) | reinterpret_cast<uintptr_t>(p.B) | row) & (kRowBytes - 1);
  if (at == 0 || ((uint64_t)p.E * b_rows * row < (64u << 20) && !p.by_lines)) return false;
  const uint64_t unit = at & (0 - at), tail = row % kRowBytes != 0 ? row % kRowBytes : kRowBytes;
  if (tail > unit && p.K <= 5 * BK && !p.by_lines) return false;
  return (uint64_t)p.M * row + 256 < (1ull << 32) && b_rows * row + 256 < (1ull << 32);   // room for the 128 bytes on top of an offset
}
// Scale rows in chunks of two pairs of stages: for experts' weights of 64 MB and more, which in a model of many layers come from HBM,
// over so many stages that the lines saved outweigh the second load of a chunk (rows of one to three chunks have none to save).
// Pairs -> chunks, 70 - 300 MB of weights, 4096 (K = 2880: 2880) weight rows, 4 / 14 (32-row tiles) and 50 / 100 rows (128-row tiles) of each
// expert, time by chunks over time by pairs:
//  * rows that start at a line, weights from HBM: K = 768 - 1536 0.99 - 1.01 (1280 beyond 256 MB 0.98 - 1.00), 1792 and 2048 0.97 - 1.00,
//    2816 0.96 - 1.00, 4096 0.94 - 1.00, 14336 0.89 - 0.97;
//  * the same weights still in the last-level cache (below 256 MB; a layer replayed alone): K = 768 - 1536 1.01 - 1.05, 2048 0.96 - 1.03,
//    4096 0.98 - 1.05, 7168 0.93 - 1.00 -- the price of the rule up to K = 4096;
//  * by lines, from HBM: 32-row tiles K = 1056 1.00 - 1.02, 1312 1.00 - 1.01, 1568 0.99 - 1.00, 2880 0.97 - 0.99; 128-row tiles K = 1056 - 1312
//    1.00 - 1.06, 1696 1.01 - 1.03, 2080 0.98 - 1.03, 2880 0.98 - 1.01, 4256 0.97 - 0.99.
// Tables of random routing, 20 - 170 rows on average: 0.92 - 1.00 (one in 64 of those calls 1.03); the same few rows behind a whole tile in every
// expert, which routing does not give, up to 1.2 (51 x 137 rows, 6656 x 6144).
template <bool SWIGLU>
bool scale_chunks(const MxArgs& p, int rows, bool lines) {
  if (p.scale_chunks != 0) return p.scale_chunks > 0;
  if (p.by_lines) return true;
  const uint64_t bytes = (uint64_t)p.E * p.N * (SWIGLU ? 2 : 1) * (uint64_t)(p.K / 2);
  if (bytes < (64u << 20)) return false;
  if (lines) return p.K > (rows == 128 ? 8 * BK : 6 * BK);
  return p.K > (bytes > (256u << 20) ? 4 * BK : 6 * BK);
}
template <bool SWIGLU, bool QUANT>
hipError_t launch_grouped(const MxArgs& p, int rows, hipStream_t s) {
  const bool lines = by_lines<SWIGLU>(p), chunks = scale_chunks<SWIGLU>(p, rows, lines);
  if (lines && chunks) return launch_grouped_lines<SWIGLU, QUANT, true, true>(p, rows, s);
  if (lines) return launch_grouped_lines<SWIGLU, QUANT, true, false>(p, rows, s);
  if (chunks) return launch_grouped_lines<SWIGLU, QUANT, false, true>(p, rows, s);
  return launch_grouped_lines<SWIGLU, QUANT, false, false>(p, rows, s);
}

// silu(gate) * up of K slices' sums P[slices][M][2N] (N gate columns, then N up columns), added up in slice order: bf16 into C, or
// (QUANT) quantised to MXFP4 with the stand-alone quantiser's steps on the bf16 values.  A lane owns 8 outputs of one row, so a block
// of 32 is four neighbouring lanes (N % 32 == 0: blocks never leave a row).  Bound by the sums' way through the memory system.
template <bool QUANT>
__global__ __launch_bounds__(256) void reduce_swiglu_kernel(MxArgs p) {
  const unsigned per_row = (unsigned)p.N / 8;
  const size_t lanes = (size_t)p.M * per_row, step = (size_t)p.M * 2 * p.N;
  const bool vec_ok = (reinterpret_cast<uintptr_t>(p.C) & 15) == 0;   // (N % 8 == 0)
  for (size_t g = (size_t)blockIdx.x * 256 + threadIdx.x; g < lanes; g += (size_t)gridDim.x * 256) {
    const size_t m = g / per_row;
    const unsigned n = (unsigned)(g % per_row) * 8;
    const float* at = p.P + m * 2 * p.N + n;
    v4f gate[2] = {}, up[2] = {};
#pragma unroll 4
    for (int sl = 0; sl < p.slices; ++sl) {
      const v4f* x = reinterpret_cast<const v4f*>(at + sl * step);
      const v4f* y = reinterpret_cast<const v4f*>(at + sl * step + p.N);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        gate[i] += x[i];
        up[i] += y[i];
      }
    }
    float hv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) hv[e] = silu(gate[e >> 2][e & 3]) * up[e >> 2][e & 3];
    const v4i o = {(int)pack_bf16x2(hv[0], hv[1]), (int)pack_bf16x2(hv[2], hv[3]), (int)pack_bf16x2(hv[4], hv[5]), (int)pack_bf16x2(hv[6], hv[7])};
    if constexpr (!QUANT) {
      uint16_t* c = p.C + m * p.N + n;
      if (vec_ok) {
        *reinterpret_cast<v4i*>(c) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) c[e] = (uint16_t)(((unsigned)o[e >> 1] >> (16 * (e & 1))) & 0xFFFF);
      }
    } else {
      float v[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[2 * j] = __builtin_bit_cast(float, (unsigned)o[j] << 16);
        v[2 * j + 1] = __builtin_bit_cast(float, (unsigned)o[j] & 0xFFFF0000u);
      }
      const int byte = mx_scale_byte(lane_xor_max_bits(lane_xor_max_bits(abs_max_bits(v), 1), 2));
      const float scale = mx_scale_value(byte);
      unsigned codes = 0;
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, v[0], v[1], scale, 0);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, v[2], v[3], scale, 1);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, v[4], v[5], scale, 2);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, v[6], v[7], scale, 3);
      *reinterpret_cast<unsigned*>(p.Q + m * (q_row_cols(p) / 2) + n / 2) = byte == 0xFF ? 0u : codes;
      if ((n & 31) == 0) p.Qs[m * (q_row_cols(p) / 32) + n / 32] = (uint8_t)byte;
    }
  }
}

// The K slices' sums of all weight rows (gate and up rows alike), then the sum over the slices.
template <int R>
hipError_t launch_split(const MxArgs& p, hipStream_t s) {
  MxArgs q = p;
  q.swiglu = 0;
  q.N = p.swiglu ? 2 * p.N : p.N;
  if (hipError_t e = launch<R, false, false, false, true, false, false>(q, s); e != hipSuccess) return e;
  if (!p.swiglu) return launch_splitk_reduce(p.P, p.C, (size_t)p.M * (size_t)p.N, p.slices, s);
  const size_t blocks = ((size_t)p.M * (p.N / 8) + 255) / 256;
  const dim3 grid((unsigned)(blocks < 4096 ? blocks : 4096));
  if (p.Q) hipLaunchKernelGGL(reduce_swiglu_kernel<true>, grid, dim3(256), 0, s, p);
  else hipLaunchKernelGGL(reduce_swiglu_kernel<false>, grid, dim3(256), 0, s, p);
  return hipGetLastError();
}
template <int R>
hipError_t launch_form(const MxArgs& p, hipStream_t s) {
  if (p.P) return launch_split<R>(p, s);
  if (p.swiglu && p.Q) return launch<R, true, true, false, false, false, false>(p, s);
  if (p.swiglu) return launch<R, true, false, false, false, false, false>(p, s);
  return launch<R, false, false, false, false, false, false>(p, s);
}

}  // namespace

// K a multiple of 32 from 512 up, 16-byte aligned A and B, 32-bit offsets over the rows of A and over one expert's weight rows,
// a tile count that fits an int.  Scale rows may start anywhere.
bool mx_stream_supports(const MxArgs& p) {
  if ((p.row_offsets ? p.E <= 0 : p.E != 0) || p.M <= 0 || p.N <= 0 || p.K < 2 * BK || p.K % 32 != 0) return false;
  if (p.Q && (!p.swiglu || !p.Qs || p.N % 32 != 0 || (reinterpret_cast<uintptr_t>(p.Q) & 3))) return false;
  if (((reinterpret_cast<uintptr_t>(p.A) | reinterpret_cast<uintptr_t>(p.B)) & 15) != 0) return false;
  const uint64_t b_rows = (uint64_t)p.N * (p.swiglu ? 2 : 1);
  if ((uint64_t)p.M * (uint64_t)(p.K / 2) >= (1ull << 32) || b_rows * (uint64_t)(p.K / 2) >= (1ull << 32)) return false;
  const uint64_t tiles = ((uint64_t)(p.M + 31) / 32 + (uint64_t)p.E) * (uint64_t)((p.N + BN / 2 - 1) / (BN / 2));
  return tiles * (uint64_t)(p.row_offsets ? 1 : p.slices) < (1ull << 30);
}

namespace {
// m-tiles of R rows that E experts with `rows` rows on average (and the spread of random routing) are expected to fill
double expected_m_tiles(int E, double rows, int R) {
  double per_expert = 1.0;
  const double sigma = sqrt(rows < 1.0 ? 1.0 : rows);
  for (int k = 1; k * R < rows + 6 * sigma; ++k) per_expert += 0.5 * erfc((k * R + 0.5 - rows) / (sigma * 1.41421356));
  return E * per_expert;
}
}  // namespace

// Shape-based dispatch; the host knows the average number of rows per expert only (what it says below 128 is the least height:
// the kernel takes taller tiles where the table is uneven, rows_for_table).  Up to 128 this kernel: it reads
// the weights once at 4 - 5.5 TB/s (gate+up of 8 experts x 16 rows, 28672 x 4096, 92 us; 128 experts x 16 rows, 5760 x 2880, 247 us where
// the 128-row tiles with a ring per tile took 318; 78 experts x 4 rows, 21504 x 1184, 205 against 306).  32 rows a tile up to 18 rows per
// expert (an expert with more rows takes a second tile and its weights a second time through the load path: 36 rows on
// average 105 us, on 64-row tiles 87 us), 64 up to 44 (64 rows on average 137 us, on 128-row tiles 111), 128 above.
// More than 128 rows per expert: against the 256 x 256 kernel, by a model of both in microseconds on 256 compute units -- 0.84 per stage and round
// here; there 2.1 - 2.8 per stage and round and 4 - 14 around a tile, more where few tiles share a weight panel or K has a tail
// (22 experts x 134 rows, 3072 x 12800: 171 us here, 220 there; 25600 x 3072: 310 here, 272 there).
int mx_stream_rows(const MxArgs& p) {
  if (!p.row_offsets || !mx_stream_supports(p)) return 0;
  const double rows = (double)p.M / p.E;
  if (rows <= 18) return 32;
  if (rows <= 44) return 64;
  if (rows <= 128) return 128;
  if (rows > 1024) return 0;
  int cus = compute_units();
  if (cus <= 0) cus = 256;
  const int stages = (p.K + BK - 1) / BK;
  const long n_here = p.swiglu ? (p.N + 63) / 64 : (p.N + 127) / 128, n_there = p.swiglu ? (p.N + 127) / 128 : (p.N + 255) / 256;
  const double here = ceil(expected_m_tiles(p.E, rows, 128) * n_here / cus) * stages * 0.84 + 4.0;
  const double m_there = expected_m_tiles(p.E, rows, 256);
  const bool whole = p.K % (2 * BK) == 0, wide = n_there >= 64;
  const double per_stage = !whole ? 2.8 : (wide ? 2.1 : 2.3), around = whole && wide ? 6.0 : (m_there < 1.3 * p.E ? 14.0 : 4.0);
  const double there = ceil(m_there * n_there / cus) * (stages * per_stage + around);
  return here < there ? 128 : 0;
}

namespace {
// The weight-streaming kernel's time in microseconds for `rows_b` weight rows (see mx_stream_plan); its fused quantiser takes whole
// blocks of 32 outputs, four tiles, to a workgroup.
double ring_us(int M, long rows_b, int K, bool quant, int cus) {
  auto ceil_div = [](long a, long b) { return (a + b - 1) / b; };
  const int mb = M <= 16 ? 0 : (M <= 32 ? 1 : 2), units = K / 512;
  const double a[3] = {3.1e-4, 3.5e-4, 4.4e-4}, b[3] = {1.35e-4, 2.8e-4, 5.4e-4};
  const int tiles = (int)ceil_div(rows_b, 16), t = quant ? tiles_per_workgroup(tiles, cus, 8, 4) : tiles_per_workgroup(tiles, cus, 7);
  const double panels = units >= 4 ? ceil_div(units, 4) * 2048.0 : units * 512.0;
  return 2.3 + ceil_div(ceil_div(tiles, t), cus) * (t * a[mb] + b[mb]) * panels + (K % 512 ? 1.2 : 0.0);
}
}  // namespace

// SwiGLU and quantiser of up to 32 rows as two launches, the bf16 form and the quantiser: where the fused quantiser's four tiles a
// workgroup leave most compute units idle.  The second launch takes 1.6 - 2.2 us; the model is good to about one.  Fused -> two
// launches: 1 x 512 x 8192 11.0 -> 6.8 us, 20 x 1536 x 5184 12.4 -> 9.0, 2 x 3072 x 7424 16.4 -> 13.1; kept fused: 4 x 4608 x 7680
// (14.6, two launches 15.1), 32 x 4096 x 4096 (9.7, 10.4), 16 x 1024 x 1024 (4.6, 5.2).
bool mx_swiglu_quant_in_two(int M, int N, int K, int cus) {
  if (cus <= 0) cus = 256;
  if (M <= 0 || M > 32 || N <= 0 || N % 32 != 0 || K < 2 * BK || K % 32 != 0) return false;
  return ring_us(M, 2L * N, K, true, cus) > ring_us(M, 2L * N, K, false, cus) + 3.0;
}

// The plain GEMM and the fused SwiGLU forms of one matrix of M rows.  The other kernels tile N alone (the weight-streaming kernel: 16
// weight rows a tile, the fused quantiser whole blocks of 32 outputs; the narrow-tile kernel 128 weight rows), so few weight rows leave
// compute units idle for the whole of K, and a K that is no multiple of 512 costs the narrow-tile kernel 5 us.  The best of them and
// of this kernel, K whole or in slices, by a model in microseconds fitted to graph replays of 72 plain shapes (1 .. 256 rows; most
// within 15 %):
//  * weight-streaming kernel: 2.3 + rounds x (tiles per workgroup x a + row blocks' b) x K in whole panels of 2048, 1.2 for a K tail;
//  * narrow-tile kernel: 3 + the larger of 0.40 - 0.47 a stage and the memory time, 5 for a K tail; 256 x 256 tiles 1.65 a stage;
//  * here: 3.3 + the larger of 0.42 - 0.5 a stage and the memory time, slices' sums 3.5 for the second launch and 7 TB/s there and back;
//  * memory time: the weights at 7 TB/s and what is read again from L2 at 16 TB/s; a third more where rows do not start at whole
//    128-byte lines.
// Measured on weights from HBM, before -> after: with a workspace 128 x 1792 x 16096 81 -> 21 us, 62 x 1792 x 16096 21.4 -> 17.1; K whole
// 128 x 9216 x 8832 40.9 -> 31.5, without a workspace 128 x 4096 x 14336 44.7 -> 36.5 and 100 x 5120 x 13824 43.6 -> 35.0 (with one both
// keep the narrow-tile kernel's slices, 19.3 and 19.8).
MxStreamPlan mx_stream_plan(int M, int N, int K, bool swiglu, bool quant, int cus, bool may_split) {
  MxStreamPlan plan;
  if (cus <= 0) cus = 256;
  if (M <= 0 || N <= 0 || K < 2 * BK || K % 32 != 0 || M > 2048 || (swiglu && N % 8 != 0)) return plan;
  // The plain GEMM of up to 64 rows (above 32: below K = 12288) gives the weight-streaming kernel's bits whether or not the
  // caller provides a workspace; its slices would save 1 - 3 us of 10 - 16 in places (32 x 5120 x 13824: 15.7 -> 12.8).
  if (!swiglu && (M <= 32 || (M <= 64 && K < 12288))) return plan;
  auto ceil_div = [](long a, long b) { return (a + b - 1) / b; };
  const long rows_b = (long)N * (swiglu ? 2 : 1);
  const double pitch = K % 256 != 0 ? 1.35 : 1.0, weights = (double)rows_b * K * 0.53;
  const int stages = (K + BK - 1) / BK, pairs = K / (2 * BK);
  auto memory = [&](double items, double item_stages, int rows_a) {
    const double all = items * item_stages * (rows_a + BN) * 136.0;
    return (weights / 7e6 + (all > weights ? all - weights : 0.0) / 16e6) * pitch;
  };
  auto larger = [](double a, double b) { return a > b ? a : b; };
  // ---- what the other kernels take --------------------------------------------------------------------------------------
  double other = 1e30;
  // Up to 32 rows both fused forms cut K alike (or not at all), so that quantising the one's result is the other, bit for bit: the
  // plan is that of the bf16 form.  Above, the weight-streaming kernel has no quantiser.
  if (M <= (quant ? 32 : 64)) other = ring_us(M, rows_b, K, false, cus);
  if (M > 32) {
    const long half = ceil_div(M, 128) * ceil_div(rows_b, 128), full = ceil_div(M, 256) * ceil_div(rows_b, 128);
    if (full <= cus) {
      const bool h = M <= 128 || half <= cus;
      const double per_stage = !h ? 0.85 : (M <= 64 ? 0.40 : 0.47);
      const double t = 3.0 + larger(stages * per_stage, memory(h ? half : full, stages, h ? (M < 128 ? M : 128) : 256)) + (K % 512 ? 5.0 : 0.0);
      other = other < t ? other : t;
    } else {
      const double t = 3.0 + ceil_div(ceil_div(M, 256) * ceil_div(rows_b, 256), cus) * stages * 1.65 + (K % 512 ? 5.0 : 0.0);
      other = other < t ? other : t;
    }
  }
  if (may_split && !swiglu) {   // the split that mx_tile_split_plan would take
    const SplitPlan split = mx_tile_split_plan_for(M, N, K, cus);
    if (split.slices > 1) {
      const double per_stage = !split.narrow ? 1.65 : (!split.half ? 0.85 : (M <= 64 ? 0.40 : 0.47));
      const long tiles = ceil_div(M, split.half ? 128 : 256) * ceil_div(N, split.narrow ? 128 : 256);
      const double t = 6.0 + larger(2 * split.slice_pairs * per_stage, memory(tiles * split.slices, 2 * split.slice_pairs, split.half ? (M < 128 ? M : 128) : 256)) +
                       8.0 * split.slices * M * N / 7e6;
      other = other < t ? other : t;
    }
  }
  // ---- this kernel ----------------------------------------------------------------------------------------------------------
  double best = other * 0.92;   // (the model is no better than that)
  for (int rows = 32; rows <= 128; rows *= 2) {
    if ((rows == 32 && M > 64) || (rows == 128 && M <= 32)) continue;
    const long tiles = ceil_div(M, rows) * ceil_div(rows_b, BN);
    const int rows_a = M < rows ? M : rows;
    const double per_stage = rows == 128 ? 0.50 : 0.42;
    const double whole = 3.3 + larger(ceil_div(tiles, cus) * stages * per_stage, memory(tiles, stages, rows_a));
    if (tiles <= cus && M > 32 && whole < best) {
      best = whole;
      plan = {rows, 1, 0, 0};
    }
    if (!may_split) continue;
    for (int want = 2; want <= pairs && tiles * want <= cus; ++want) {
      const int per = (int)ceil_div(pairs, want);
      if (ceil_div(pairs, per) != want) continue;
      const double sums = 4.0 * want * M * rows_b;
      const double item_stages = 2.0 * per + (K % 512) / 256.0;
      const double t = 6.8 + larger(item_stages * per_stage, memory(tiles * want, item_stages, rows_a)) + 2.0 * sums / 7e6;
      if (t < best) {
        best = t;
        plan = {rows, want, per, (size_t)want * (size_t)M * (size_t)rows_b * sizeof(float)};
      }
    }
  }
  return plan;
}

hipError_t launch_mx_stream(const MxArgs& p, int tile_rows, hipStream_t s) {
  if (p.row_offsets) {
    if (p.swiglu && p.Q) return launch_grouped<true, true>(p, tile_rows, s);
    if (p.swiglu) return launch_grouped<true, false>(p, tile_rows, s);
    return launch_grouped<false, false>(p, tile_rows, s);
  }
  return tile_rows == 32 ? launch_form<32>(p, s) : (tile_rows == 64 ? launch_form<64>(p, s) : launch_form<128>(p, s));
}

}  // namespace ave
