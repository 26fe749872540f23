// The two steps in front of the grouped (MoE) GEMM, on the device so that the whole expert layer can
// be recorded into one HIP graph:
//
//   route_choose_kernel, route_place_kernel
//                       router logits [T, E] -> for every token its two highest-scoring experts, the
//                       2T routed rows sorted by expert (stable: by token, then by rank) as a list of
//                       token indices, the E+1 row offsets the grouped GEMM reads, and the softmax
//                       probability of every routed row;
//   gather_rows_kernel  packed MXFP4 rows and their scale rows copied into that order;
//   combine_top2_kernel the step behind the expert GEMMs: every token's two expert outputs, weighted with their
//                       routing probabilities, summed back into token order.
//
// Routing is a counting sort over chunks of tokens.  The tokens' choices are found once, by subgroups of lanes that read
// a row of logits coalesced; a chunk's rows start where the experts below and the chunks before it end, and inside a chunk
// up to 1024 tokens at a time are ranked with ballots over the bits of the expert numbers.  Tokens rise with (chunk, block of
// 1024, wave, lane), so the order inside an expert is by token: the stable order.  A few tokens are one launch of one
// workgroup; more tokens are two launches that pass the choices and the chunks' counts through a workspace, or, without
// one, a single launch in which every workgroup counts all tokens.
#include "fp4_common.hpp"
#include "kernels.hpp"

namespace ave {
namespace {

constexpr int kRouteThreads = 1024;
constexpr int kRouteBlock = kRouteThreads;   // tokens that are ranked together at most, one a thread
constexpr int kRouteChunk = 256;       // tokens of a workgroup where there are several (more only for the largest T)
constexpr int kRouteMaxE = 256;
constexpr int kRouteMaxChunks = 256;
constexpr int kRoutePartsMax = 32;     // workgroups that go through all tokens
constexpr int kRouteValues = 8;        // logits of one token that a lane holds

// Bound by latency: a few dependent trips to memory per kernel, and what one compute unit computes in between.  With a workspace
// every token's logits are read once: 16384 tokens and 8 experts 8.4 us, 2443 tokens and 141 experts 11.5 us.  Without one every workgroup goes
// through all tokens (count_all): 20.7 and 84 us, 131072 tokens and 8 experts 122 us (one workgroup per expert and eighth of the
// tokens, each with a plain scan: 24, 288 and 163 us; 512 to 2048 tokens and 8 experts 6.8 - 9.0 us then, 7.6 - 10.3 us now).
// A chunk is what one workgroup takes: the tokens whose choices it finds in one go (1024 lanes, E / 8 of them per token, at
// most 256 tokens), and never more than 256 chunks, so that a workgroup's sum over the chunks before it stays a few loads per
// thread.  Up to two goes and 512 tokens stay with one workgroup: the second costs about what the second launch would.
struct RouteShape {
  int lanes_log2;                // lanes per token: the power of two from E / 8 up
  int chunk_tokens, chunks;
};
inline RouteShape route_shape(int T, int E) {
  RouteShape r{0, 0, 1};
  while ((kRouteValues << r.lanes_log2) < E) ++r.lanes_log2;
  const int go = kRouteThreads >> r.lanes_log2;
  const int least = (T + kRouteMaxChunks - 1) / kRouteMaxChunks, chunk = go < kRouteChunk ? go : kRouteChunk;
  r.chunk_tokens = chunk > least ? chunk : least;
  if (T <= 2 * go && T <= 512) r.chunk_tokens = kRouteBlock;
  r.chunks = T > 0 ? (T + r.chunk_tokens - 1) / r.chunk_tokens : 1;
  return r;
}

struct RouteArgs {
  const float* logits;
  int T, E;
  int lanes_log2;
  int chunk_tokens, chunks;
  int32_t* token_of_row;
  int32_t* row_offsets;
  float* row_weight;             // may be null
  int32_t* rows_of_token;        // may be null: [T, 2], the routed row of every token's first and second choice
  int* counts;                   // workspace: [chunks][E] routed rows, ...
  unsigned* pairs;               // ... [T] first choice | second choice << 16,
  v2f* probs;                    // ... [T] their probabilities
};

struct Choice {
  float v;   // not NaN
  int e;     // -1: none, v is minus infinity
};
// Among equal scores the lower expert index.
__device__ inline bool ranks_before(const Choice& a, const Choice& b) { return a.v > b.v || (a.v == b.v && a.e < b.e); }

// A token's logits as its subgroup of lanes holds them: lane `sub` of L those of experts sub, sub + L, ...
__device__ inline void load_logits(const RouteArgs& p, int t, int sub, int L, float (&x)[kRouteValues]) {
  const float* l = p.logits + (size_t)t * p.E;
#pragma unroll
  for (int j = 0; j < kRouteValues; ++j) {
    const int e = j * L + sub;
    x[j] = e < p.E ? l[e] : -__builtin_inff();
  }
}

// The choices of one token by a scan over the experts that starts with experts 0 and 1 and replaces a choice only by a greater score.
// So a NaN never hides the finite logits: that of expert 0 stays the first choice, that of expert 1 the second behind expert
// 0, any other is passed over.
__device__ inline void scan_token(const float* l, int E, Choice& first, Choice& second) {
  int a = 0, b = -1;
  for (int e = 1; e < E; ++e) {
    if (l[e] > l[a]) {
      b = a;
      a = e;
    } else if (b < 0 || l[e] > l[b]) {
      b = e;
    }
  }
  first = {l[a], a};
  second = {l[b], b};
}

// Puts the logit of expert e, which is behind those that were put before it, among a lane's first and second choice.  Two comparisons
// that leave NaN and minus infinity out: where these could matter the token is scanned.
__device__ inline void put(float v, int e, Choice& first, Choice& second) {
  const bool better = v > first.v, next = v > second.v;
  second.v = better ? first.v : (next ? v : second.v);
  second.e = better ? first.e : (next ? e : second.e);
  first.v = better ? v : first.v;
  first.e = better ? e : first.e;
}
// The choices of a subgroup of L lanes from those of its lanes
__device__ inline void merge(int L, Choice& first, Choice& second) {
  for (int d = 1; d < L; d <<= 1) {
    const Choice f{__shfl_xor(first.v, d, 64), __shfl_xor(first.e, d, 64)};
    const Choice s{__shfl_xor(second.v, d, 64), __shfl_xor(second.e, d, 64)};
    const bool better = ranks_before(f, first);
    // the second of both is the loser of the two firsts or the winner's own second
    const Choice lost = better ? first : f, own = better ? s : second;
    first = better ? f : first;
    second = ranks_before(lost, own) ? lost : own;
  }
}

// The choices of `n` tokens (at most kRouteBlock) from token `t0` on, into pair[] and, when wanted, prob[] (both LDS): the two
// experts and their probabilities in the full softmax.
// The softmax denominator is added up in double: a float sum of E terms drifts by about sqrt(E) roundings, which for 200 and more experts is more than the
// 2e-6 relative error the probabilities are stated to keep.  Its terms take expf: v_exp_f32 on x log2(e) is off by
// |x| 2^-24 where that product is rounded, which shows in the sum of 64 and more (rms error of the probabilities, 64 .. 256
// experts: 3.4 - 3.6e-8, with expf 3.0e-8), and the kernel waits for memory either way.
__device__ inline void choose_block(const RouteArgs& p, int t0, int n, bool want_prob, unsigned* pair, v2f* prob) {
  const int L = 1 << p.lanes_log2, sub = threadIdx.x & (L - 1);
  for (int i = threadIdx.x >> p.lanes_log2; i < n; i += kRouteThreads >> p.lanes_log2) {
    float x[kRouteValues];
    load_logits(p, t0 + i, sub, L, x);
    Choice first{-__builtin_inff(), -1}, second{-__builtin_inff(), -1};
#pragma unroll
    for (int j = 0; j < kRouteValues; ++j)
      if (j * L < p.E) put(x[j], j * L + sub, first, second);
    merge(L, first, second);
    // a NaN of expert 0 or 1, or fewer than two logits above minus infinity (the whole subgroup takes the branch)
    const bool nan = L == 1 ? x[0] != x[0] || x[1] != x[1] : sub < 2 && x[0] != x[0];
    const unsigned long long odd = __ballot(nan || second.e < 0), group = ((1ull << L) - 1) << (threadIdx.x & 63 & ~(L - 1));
    if (odd & group) scan_token(p.logits + (size_t)(t0 + i) * p.E, p.E, first, second);
    if (want_prob) {
      double sum = 0.0;
#pragma unroll
      for (int j = 0; j < kRouteValues; ++j) {   // (the first choice's own term is 1 also where it is an infinity)
        if (j * L >= p.E) break;
        const float d = j * L + sub == first.e && x[j] == x[j] ? 0.f : x[j] - first.v;
        sum += (double)expf(j * L + sub < p.E ? d : -__builtin_inff());
      }
      for (int d = 1; d < L; d <<= 1) sum += __shfl_xor(sum, d, 64);
      if (sub == 0) prob[i] = v2f{(float)(1.0 / sum), (float)((double)expf(second.v - first.v) / sum)};
    }
    if (sub == 0) pair[i] = (unsigned)first.e | (unsigned)second.e << 16;
  }
}

// The sum over a wave's lanes, in lane 63
__device__ inline unsigned wave_sum(unsigned v) {
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true);   // row_shr:1, 2, 4, 8: lane 15 of a row has its sum
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, true);
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, true);
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, true);
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);  // row_bcast15 into rows 1 and 3
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);  // row_bcast31 into rows 2 and 3
  return v;
}

// Adds the routed rows per expert of all tokens to total[], those of the tokens in front of t_begin to before[] (both LDS).
// Bound by the instructions of one compute unit, since every workgroup does this for itself: a lane takes up to 32 logits of a token,
// four neighbours at a time and the next trip's under way, and scans them with two comparisons each that leave NaN and minus infinity out;
// a token that these could matter to is scanned again.  No barrier; where there are few experts (E <= 8) counters in registers instead
// of 64 atomics on a few addresses.
template <int kGroups>   // of four logits; 2 for up to 8 experts
__device__ inline void count_all(const RouteArgs& p, int t_begin, int* total, int* before) {
  int lanes_log2 = 0;          // lanes per token: 1 up to 32 experts, 8 for 256
  while ((4 * kGroups << lanes_log2) < p.E) ++lanes_log2;
  const int L = 1 << lanes_log2, sub = threadIdx.x & (L - 1), step = kRouteThreads >> lanes_log2;
  const int groups = (p.E + 4 * L - 1) / (4 * L);
  const bool vec = (p.E & 3) == 0 && (reinterpret_cast<uintptr_t>(p.logits) & 15) == 0;
  constexpr bool packed = kGroups == 2;   // an expert's rows in a byte of its own, per lane
  unsigned long long rows = 0, rows_before = 0;
  auto flush = [&]() {   // the wave's bytes added up: fields of 16 bits hold 64 x 255
    unsigned field[8];   // experts {0, 2} {4, 6} {1, 3} {5, 7} of all tokens, then of those before
#pragma unroll
    for (int i = 0; i < 8; ++i) field[i] = (unsigned)((i < 4 ? rows : rows_before) >> (i & 2 ? 8 : 0) >> (i & 1 ? 32 : 0)) & 0x00FF00FFu;
#pragma unroll
    for (int i = 0; i < 8; ++i) field[i] = wave_sum(field[i]);
    if ((threadIdx.x & 63) == 63) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int i = e / 4 + 2 * (e & 1), shift = 16 * (e >> 1 & 1);
        atomicAdd(&total[e], (int)(field[i] >> shift & 0xFFFF));
        atomicAdd(&before[e], (int)(field[i + 4] >> shift & 0xFFFF));
      }
    }
    rows = rows_before = 0;
  };
  v4f x[kGroups], ahead[kGroups];
  const v4f none = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
  auto load = [&](int t, v4f (&to)[kGroups]) {
    const float* l = p.logits + (size_t)(t < p.T ? t : p.T - 1) * p.E;
#pragma unroll
    for (int j = 0; j < kGroups; ++j) {
      if (j >= groups) break;
      const int e = (j * L + sub) * 4;
      to[j] = none;
      if (vec) {
        if (e < p.E) to[j] = *reinterpret_cast<const v4f*>(l + e);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (e + q < p.E) to[j][q] = l[e + q];
      }
    }
  };
  int t = threadIdx.x >> lanes_log2, trips = 0;
  load(t, x);
  for (int t0 = 0; t0 < p.T; t0 += step, t += step) {   // the same trips for all lanes
    if (t0 + step < p.T) load(t + step, ahead);
    Choice first{-__builtin_inff(), -1}, second{-__builtin_inff(), -1};
#pragma unroll
    for (int j = 0; j < kGroups; ++j) {
      if (j >= groups) break;
#pragma unroll
      for (int q = 0; q < 4; ++q) put(x[j][q], (j * L + sub) * 4 + q, first, second);
    }
    merge(L, first, second);
    const bool on = t < p.T && sub == 0;
    if (on && (second.e < 0 || x[0][0] != x[0][0] || x[0][1] != x[0][1])) scan_token(p.logits + (size_t)t * p.E, p.E, first, second);
    if constexpr (packed) {
      const unsigned long long one = on ? (1ull << (8 * first.e)) + (1ull << (8 * second.e)) : 0;
      rows += one;
      rows_before += t < t_begin ? one : 0;
      if (++trips == 255) {
        flush();
        trips = 0;
      }
    } else if (on) {
      atomicAdd(&total[first.e], 1);
      atomicAdd(&total[second.e], 1);
      if (t < t_begin) {
        atomicAdd(&before[first.e], 1);
        atomicAdd(&before[second.e], 1);
      }
    }
#pragma unroll
    for (int j = 0; j < kGroups; ++j)
      if (j < groups) x[j] = ahead[j];
  }
  if (packed) flush();
}

// First of the two launches: a chunk's choices and its routed rows per expert, into the workspace.
__global__ __launch_bounds__(kRouteThreads) void route_choose_kernel(RouteArgs p) {
  __shared__ unsigned pair[kRouteBlock];
  __shared__ v2f prob[kRouteBlock];
  __shared__ int count[kRouteMaxE];
  const int tid = threadIdx.x;
  const int t_begin = blockIdx.x * p.chunk_tokens;
  const int t_end = t_begin + p.chunk_tokens < p.T ? t_begin + p.chunk_tokens : p.T;
  if (tid < kRouteMaxE) count[tid] = 0;
  for (int t0 = t_begin; t0 < t_end; t0 += kRouteBlock) {
    const int n = t_end - t0 < kRouteBlock ? t_end - t0 : kRouteBlock;
    choose_block(p, t0, n, p.row_weight != nullptr, pair, prob);
    __syncthreads();
    if (tid < n) {
      const unsigned c = pair[tid];
      p.pairs[t0 + tid] = c;
      if (p.row_weight) p.probs[t0 + tid] = prob[tid];
      atomicAdd(&count[c & 0xFFFF], 1);
      atomicAdd(&count[c >> 16], 1);
    }
    __syncthreads();
  }
  if (tid < p.E) p.counts[(size_t)blockIdx.x * p.E + tid] = count[tid];
}

// Places the rows of one chunk per workgroup.  CHOSEN: choices and counts come from the workspace; otherwise the
// workgroup makes them itself, for all tokens (there is one chunk, or the caller gave no workspace).
template <bool CHOSEN>
__global__ __launch_bounds__(kRouteThreads) void route_place_kernel(RouteArgs p) {
  __shared__ unsigned pair[kRouteBlock];
  __shared__ v2f prob[kRouteBlock];
  __shared__ int before[kRouteMaxE], total[kRouteMaxE];   // rows of an expert in the chunks before this one; in all
  __shared__ int next[kRouteMaxE];                        // where an expert's next row goes
  __shared__ int of_wave[kRouteBlock / 64][kRouteMaxE];
  __shared__ int wave_total[kRouteMaxE / 64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int t_begin = blockIdx.x * p.chunk_tokens;
  const int t_end = t_begin + p.chunk_tokens < p.T ? t_begin + p.chunk_tokens : p.T;

  // of_wave[][] of the first `waves` waves to zero
  auto clear = [&](int waves) {
    for (int i = tid; i < waves * kRouteMaxE; i += kRouteThreads) of_wave[i / kRouteMaxE][i % kRouteMaxE] = 0;
  };
  // Token t0 + tid's experts and its rows' ranks among those of its wave; the wave's rows per expert into of_wave[].
  int expert[2] = {0, 0}, rank[2] = {0, 0};
  v2f weight = {0.f, 0.f};
  bool on = false;
  auto rank_rows = [&](int t0, int n) {
    on = tid < n;
    if (w >= (n + 63) / 64) return;
    unsigned c = 0;
    if (on) {
      c = CHOSEN ? p.pairs[t0 + tid] : pair[tid];
      if (p.row_weight) weight = CHOSEN ? p.probs[t0 + tid] : prob[tid];
    }
    expert[0] = (int)(c & 0xFFFF);
    expert[1] = (int)(c >> 16);
    // lanes whose token goes to expert x, as first or as second choice: bits of their expert numbers against x's
    unsigned long long same[2][2];
    const unsigned long long live = __ballot(on);
#pragma unroll
    for (int k = 0; k < 2; ++k) same[k][0] = same[k][1] = live;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      if (1 << b >= p.E) break;
      const unsigned long long has[2] = {__ballot((expert[0] >> b) & 1), __ballot((expert[1] >> b) & 1)};
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const bool bit = (expert[k] >> b) & 1;
#pragma unroll
        for (int j = 0; j < 2; ++j) same[k][j] &= bit ? has[j] : ~has[j];
      }
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const unsigned long long all = same[k][0] | same[k][1];
      rank[k] = __popcll(all & ((1ull << lane) - 1ull));
      if (on && rank[k] == 0) of_wave[w][expert[k]] = __popcll(all);
    }
  };

  if (tid < kRouteMaxE) before[tid] = total[tid] = 0;
  __syncthreads();
  if constexpr (CHOSEN) {
    // thread = (group of chunks, expert): a table row of counts is read coalesced
    int width = 1;
    while (width < p.E) width <<= 1;
    const int e = tid & (width - 1);
    if (e < p.E) {
      int sum_before = 0, sum = 0;
#pragma unroll 8
      for (int c = tid / width; c < p.chunks; c += kRouteThreads / width) {
        const int v = p.counts[(size_t)c * p.E + e];
        sum += v;
        sum_before += c < (int)blockIdx.x ? v : 0;
      }
      if (sum) atomicAdd(&total[e], sum);
      if (sum_before) atomicAdd(&before[e], sum_before);
    }
    __syncthreads();
  } else if (p.chunks == 1) {   // at most kRouteBlock tokens: ranked at once, the counts of the waves are what there is in all
    const int waves = (p.T + 63) / 64;
    clear(waves);
    choose_block(p, 0, p.T, p.row_weight != nullptr, pair, prob);
    __syncthreads();
    rank_rows(0, p.T);
    __syncthreads();
    if (tid < kRouteMaxE)
      for (int ww = 0; ww < waves; ++ww) total[tid] += of_wave[ww][tid];
  } else {
    if (p.E <= 8) count_all<2>(p, t_begin, total, before);
    else count_all<8>(p, t_begin, total, before);
    __syncthreads();
  }

  // exclusive sum of the totals over the experts
  if (tid < kRouteMaxE) {
    const int mine = total[tid];
    int run = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(run, d, 64);
      run += lane >= d ? o : 0;
    }
    if (lane == 63) wave_total[w] = run;
    next[tid] = run - mine;
  }
  __syncthreads();
  if (tid < kRouteMaxE) {
    int start = next[tid];
    for (int ww = 0; ww < w; ++ww) start += wave_total[ww];
    if (blockIdx.x == 0 && tid < p.E) {
      p.row_offsets[tid + 1] = start + total[tid];
      if (tid == 0) p.row_offsets[0] = 0;
    }
    next[tid] = start + before[tid];
  }

  for (int t0 = t_begin; t0 < t_end; t0 += kRouteBlock) {
    const int n = t_end - t0 < kRouteBlock ? t_end - t0 : kRouteBlock, waves = (n + 63) / 64;
    if (CHOSEN || p.chunks > 1) {
      if constexpr (!CHOSEN) {
        __syncthreads();
        choose_block(p, t0, n, p.row_weight != nullptr, pair, prob);
      }
      clear(waves);
      __syncthreads();
      rank_rows(t0, n);
    }
    __syncthreads();
    if (on) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        int pos = next[expert[k]] + rank[k];
        for (int w0 = 0; w0 < w; w0 += 4)   // four reads under way (rows behind wave w - 1: of other waves, or not written; not added)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int v = of_wave[w0 + j][expert[k]];
            pos += w0 + j < w ? v : 0;
          }
        p.token_of_row[pos] = t0 + tid;
        if (p.row_weight) p.row_weight[pos] = weight[k];
        if (p.rows_of_token) p.rows_of_token[2 * (size_t)(t0 + tid) + k] = pos;
      }
    }
    __syncthreads();
    if (tid < kRouteMaxE)
      for (int ww = 0; ww < waves; ++ww) next[tid] += of_wave[ww][tid];
    __syncthreads();
  }
}

// dst row i = src row index[i] (data: row_bytes, a multiple of 16; scales: row_scales bytes moved SV at a
// time).  An index outside [0, src_rows) yields a row of zeros.  A thread moves kGatherUnroll pieces
// per trip and issues all their loads (index, then data) before the first store.
constexpr int kGatherUnroll = 4;

template <int SV>
__global__ __launch_bounds__(256) void gather_rows_kernel(const uint8_t* src, const uint8_t* src_s,
                                                          const int32_t* index, int rows, int src_rows,
                                                          unsigned row_bytes, unsigned row_scales, uint8_t* dst,
                                                          uint8_t* dst_s) {
  const unsigned data_units = row_bytes / 16, scale_units = row_scales / SV, units = data_units + scale_units;
  const size_t total = (size_t)rows * units, stride = (size_t)gridDim.x * 256;
  for (size_t i0 = (size_t)blockIdx.x * 256 + threadIdx.x; i0 < total; i0 += stride * kGatherUnroll) {
    unsigned row[kGatherUnroll], u[kGatherUnroll];
    int from[kGatherUnroll];
#pragma unroll
    for (int j = 0; j < kGatherUnroll; ++j) {
      const size_t i = i0 + (size_t)j * stride;
      row[j] = (unsigned)(i / units);
      u[j] = (unsigned)(i % units);
      from[j] = i < total ? index[row[j]] : -1;
    }
    v4i data[kGatherUnroll];
#pragma unroll
    for (int j = 0; j < kGatherUnroll; ++j) {
      const bool ok = from[j] >= 0 && from[j] < src_rows;
      data[j] = v4i{0, 0, 0, 0};
      if (ok) {
        if (u[j] < data_units) {
          data[j] = *reinterpret_cast<const v4i*>(src + (size_t)from[j] * row_bytes + 16 * u[j]);
        } else {
          const uint8_t* s = src_s + (size_t)from[j] * row_scales + (u[j] - data_units) * SV;
          if (SV == 16) data[j] = *reinterpret_cast<const v4i*>(s);
          else if (SV == 4) data[j][0] = *reinterpret_cast<const int*>(s);
          else data[j][0] = *s;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < kGatherUnroll; ++j) {
      if (i0 + (size_t)j * stride < total) {
        if (u[j] < data_units) {
          *reinterpret_cast<v4i*>(dst + (size_t)row[j] * row_bytes + 16 * u[j]) = data[j];
        } else {
          uint8_t* d = dst_s + (size_t)row[j] * row_scales + (u[j] - data_units) * SV;
          if (SV == 16) *reinterpret_cast<v4i*>(d) = data[j];
          else if (SV == 4) *reinterpret_cast<int*>(d) = data[j][0];
          else *d = (uint8_t)data[j][0];
        }
      }
    }
  }
}

// out[t, :] = w0 * rows[r0, :] + w1 * rows[r1, :] with (r0, r1) = rows_of_token[t] and (w0, w1) their routing
// probabilities, divided by their sum when `renormalize`.  bf16 in and out; the two products and the sum are
// single IEEE fp32 operations (no contraction into an fma), so the result does not depend on the compiler and
// equals the same three numpy float32 operations bit for bit.  A thread moves 8 columns (16 bytes) of one token.
__global__ __launch_bounds__(256) void combine_top2_kernel(const uint16_t* rows, const int32_t* rows_of_token,
                                                           const float* row_weight, int T, int H8, int n_rows,
                                                           int renormalize, uint16_t* out) {
#pragma clang fp contract(off)   // hipcc contracts a * b + c into an fma by default; the operators below are written out
                                 // (not __fmul_rn / __fadd_rn, whose bodies the pragma does not reach) so that it applies
  const size_t total = (size_t)T * H8, stride = (size_t)gridDim.x * 256;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += stride) {
    const size_t t = i / H8;
    const unsigned c = (unsigned)(i % H8);
    const int r0 = rows_of_token[2 * t], r1 = rows_of_token[2 * t + 1];
    const bool ok0 = r0 >= 0 && r0 < n_rows, ok1 = r1 >= 0 && r1 < n_rows;   // a row out of range counts as zeros
    float w0 = ok0 ? row_weight[r0] : 0.f, w1 = ok1 ? row_weight[r1] : 0.f;
    if (renormalize) {
      const float sum = w0 + w1;
      w0 = __fdiv_rn(w0, sum);
      w1 = __fdiv_rn(w1, sum);
    }
    const v4i zero = {0, 0, 0, 0};
    const v4i x0 = ok0 ? reinterpret_cast<const v4i*>(rows + (size_t)r0 * H8 * 8)[c] : zero;
    const v4i x1 = ok1 ? reinterpret_cast<const v4i*>(rows + (size_t)r1 * H8 * 8)[c] : zero;
    v4i o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a_lo = __builtin_bit_cast(float, (unsigned)x0[j] << 16), a_hi = __builtin_bit_cast(float, (unsigned)x0[j] & 0xFFFF0000u);
      const float b_lo = __builtin_bit_cast(float, (unsigned)x1[j] << 16), b_hi = __builtin_bit_cast(float, (unsigned)x1[j] & 0xFFFF0000u);
      const float lo = w0 * a_lo + w1 * b_lo;   // three roundings each: see the pragma above
      const float hi = w0 * a_hi + w1 * b_hi;
      o[j] = (int)pack_bf16x2(lo, hi);
    }
    reinterpret_cast<v4i*>(out + t * H8 * 8)[c] = o;
  }
}

}  // namespace

int route_top2_max_experts() { return kRouteMaxE; }

// [chunks][E] counts, then [T] probabilities (8 bytes), then [T] choices
size_t route_top2_workspace_bytes(int T, int E) {
  const RouteShape r = route_shape(T, E);
  if (r.chunks <= 1) return 0;
  return ((size_t)r.chunks * E * sizeof(int) + 15) / 16 * 16 + (size_t)T * (sizeof(v2f) + sizeof(unsigned));
}

hipError_t launch_route_top2(const float* logits, int T, int E, int32_t* token_of_row, int32_t* row_offsets,
                             float* row_weight, int32_t* rows_of_token, void* workspace, hipStream_t s) {
  const RouteShape r = route_shape(T, E);
  RouteArgs p{logits, T, E, r.lanes_log2, r.chunk_tokens, r.chunks, token_of_row, row_offsets, row_weight, rows_of_token, nullptr, nullptr, nullptr};
  if (r.chunks > 1 && workspace) {
    uint8_t* at = static_cast<uint8_t*>(workspace);
    p.counts = reinterpret_cast<int*>(at);
    at += ((size_t)r.chunks * E * sizeof(int) + 15) / 16 * 16;
    p.probs = reinterpret_cast<v2f*>(at);
    p.pairs = reinterpret_cast<unsigned*>(at + (size_t)T * sizeof(v2f));
    hipLaunchKernelGGL(route_choose_kernel, dim3((unsigned)r.chunks), dim3(kRouteThreads), 0, s, p);
    hipLaunchKernelGGL(route_place_kernel<true>, dim3((unsigned)r.chunks), dim3(kRouteThreads), 0, s, p);
    return hipGetLastError();
  }
  if (r.chunks > 1) {   // every workgroup goes through all tokens and places its part of them
    const int parts = r.chunks < kRoutePartsMax ? r.chunks : kRoutePartsMax;
    p.chunk_tokens = (T + parts - 1) / parts;
    p.chunks = (T + p.chunk_tokens - 1) / p.chunk_tokens;
  }
  hipLaunchKernelGGL(route_place_kernel<false>, dim3((unsigned)p.chunks), dim3(kRouteThreads), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_combine_top2(const uint16_t* rows, const int32_t* rows_of_token, const float* row_weight, int T, int H,
                               int n_rows, int renormalize, uint16_t* out, hipStream_t s) {
  const size_t total = (size_t)T * (H / 8);
  if (total == 0) return hipSuccess;
  size_t blocks = (total + 255) / 256;
  if (blocks > 256 * 16) blocks = 256 * 16;   // grid-stride beyond 16 workgroups per CU
  hipLaunchKernelGGL(combine_top2_kernel, dim3((unsigned)blocks), dim3(256), 0, s, rows, rows_of_token, row_weight, T,
                     H / 8, n_rows, renormalize, out);
  return hipGetLastError();
}

hipError_t launch_gather_rows(const uint8_t* src, const uint8_t* src_s, const int32_t* index, int rows, int src_rows,
                              int K, uint8_t* dst, uint8_t* dst_s, hipStream_t s) {
  const unsigned row_bytes = (unsigned)K / 2, row_scales = (unsigned)K / 32;
  const uintptr_t sbits = reinterpret_cast<uintptr_t>(src_s) | reinterpret_cast<uintptr_t>(dst_s) | row_scales;
  const int sv = (sbits & 15) == 0 ? 16 : ((sbits & 3) == 0 ? 4 : 1);
  const size_t total = (size_t)rows * (row_bytes / 16 + row_scales / sv);
  size_t blocks = (total + 255) / 256;
  if (blocks > 256 * 16) blocks = 256 * 16;   // grid-stride beyond 16 workgroups per CU
  const dim3 grid((unsigned)blocks), block(256);
  if (sv == 16)
    hipLaunchKernelGGL(gather_rows_kernel<16>, grid, block, 0, s, src, src_s, index, rows, src_rows, row_bytes,
                       row_scales, dst, dst_s);
  else if (sv == 4)
    hipLaunchKernelGGL(gather_rows_kernel<4>, grid, block, 0, s, src, src_s, index, rows, src_rows, row_bytes,
                       row_scales, dst, dst_s);
  else
    hipLaunchKernelGGL(gather_rows_kernel<1>, grid, block, 0, s, src, src_s, index, rows, src_rows, row_bytes,
                       row_scales, dst, dst_s);
  return hipGetLastError();
}

}  // namespace ave
