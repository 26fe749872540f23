// The two steps in front of the grouped (MoE) GEMM, on the device so that the whole expert layer can
// be recorded into one HIP graph:
//
//   route_top2_kernel   router logits [T, E] -> for every token its two highest-scoring experts, the
//                       2T routed rows sorted by expert (stable: by token, then by rank) as a list of
//                       token indices, the E+1 row offsets the grouped GEMM reads, and the softmax
//                       probability of every routed row;
//   gather_rows_kernel  packed MXFP4 rows and their scale rows copied into that order;
//   combine_top2_kernel the step behind the expert GEMMs: every token's two expert outputs, weighted with their
//                       routing probabilities, summed back into token order.
//
// Routing is a counting sort over chunks of tokens.  The tokens' choices are found once, by subgroups of lanes that read
// a row of logits coalesced; a chunk's rows start where the experts below and the chunks before it end, and inside a chunk
// 256 tokens at a time are ranked with ballots over the bits of the expert numbers.  Tokens rise with (chunk, block of
// 256, wave, lane), so the order inside an expert is by token: the stable order.  A few tokens are one launch of one
// workgroup; more tokens are two launches that pass the choices and the chunks' counts through a workspace, or, without
// one, a single launch in which every workgroup counts all tokens.
#include "fp4_common.hpp"
#include "kernels.hpp"

namespace ave {
namespace {

constexpr int kRouteThreads = 1024;
constexpr int kRouteBlock = 256;       // tokens that are ranked together
constexpr int kRouteMaxE = 256;
constexpr int kRouteMaxChunks = 256;
constexpr int kRouteValues = 8;        // logits of one token that a lane holds

// Bound by latency: a few dependent trips to memory per kernel.  Every token's logits are read once (a version whose
// workgroups -- one per expert -- each went through all tokens took 368 us for 2443 tokens and 141 experts and 27 us for
// 16384 tokens and 8 experts; the two launches below 12 us and 9.7 us).  A chunk is what one workgroup takes: the tokens whose choices it
// finds in one go (1024 lanes, E / 8 of them per token, at most 256 tokens), and never more than 256 chunks, so that a
// workgroup's sum over the chunks before it stays a few loads per thread.  Up to two goes stay with one workgroup: the
// second costs about what the second launch would.
struct RouteShape {
  int lanes_log2;                // lanes per token: the power of two from E / 8 up
  int chunk_tokens, chunks;
};
inline RouteShape route_shape(int T, int E) {
  RouteShape r{0, 0, 1};
  while ((kRouteValues << r.lanes_log2) < E) ++r.lanes_log2;
  const int go = (kRouteThreads >> r.lanes_log2) < kRouteBlock ? kRouteThreads >> r.lanes_log2 : kRouteBlock;
  const int least = (T + kRouteMaxChunks - 1) / kRouteMaxChunks;
  r.chunk_tokens = go > least ? go : least;
  if (T <= 2 * go && T <= kRouteBlock) r.chunk_tokens = kRouteBlock;
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
  float v;
  int e;   // -1: none
};
// Among equal scores the lower expert index; no order over NaN, which must not become a choice's v.
__device__ inline bool ranks_before(const Choice& a, const Choice& b) {
  return a.e >= 0 && (b.e < 0 || a.v > b.v || (a.v == b.v && a.e < b.e));
}

// The choices of `n` tokens (at most 256) from token `t0` on, into pair[] and, when wanted, prob[] (both LDS):
// highest and second-highest logit and their probabilities in the full softmax.  A NaN never hides the finite logits: the
// choices are those of a scan over the experts that starts with experts 0 and 1 and replaces a choice only by a greater
// score -- a NaN of expert 0 stays the first choice, one of expert 1 the second behind expert 0, any other is passed over.
// The softmax denominator is added up in double: a float sum of E terms drifts by about sqrt(E) roundings, which for 200 and more experts is more than the
// 2e-6 relative error the probabilities are stated to keep.  Its terms take expf: v_exp_f32 on x log2(e) is off by
// |x| 2^-24 where that product is rounded, which shows in the sum of 64 and more (rms error of the probabilities, 64 .. 256
// experts: 3.4 - 3.6e-8, with expf 3.0e-8), and the kernel waits for memory either way.
__device__ inline void choose_block(const RouteArgs& p, int t0, int n, bool want_prob, unsigned* pair, v2f* prob) {
  const int L = 1 << p.lanes_log2, sub = threadIdx.x & (L - 1);
  for (int i = threadIdx.x >> p.lanes_log2; i < n; i += kRouteThreads >> p.lanes_log2) {
    const float* l = p.logits + (size_t)(t0 + i) * p.E;
    float x[kRouteValues];
#pragma unroll
    for (int j = 0; j < kRouteValues; ++j) {
      const int e = j * L + sub;
      x[j] = e < p.E ? l[e] : 0.f;
    }
    Choice first{0.f, -1}, second{0.f, -1};
#pragma unroll
    for (int j = 0; j < kRouteValues; ++j) {   // selects, no branches
      const int e = j * L + sub;
      const bool nan = x[j] != x[j];
      const Choice c{nan ? __builtin_inff() : x[j], e < p.E && (!nan || e == 0) ? e : -1};
      const bool better = ranks_before(c, first), next = ranks_before(c, second);
      second.v = better ? first.v : (next ? c.v : second.v);
      second.e = better ? first.e : (next ? c.e : second.e);
      first.v = better ? c.v : first.v;
      first.e = better ? c.e : first.e;
    }
    for (int d = 1; d < L; d <<= 1) {
      const Choice f{__shfl_xor(first.v, d, 64), __shfl_xor(first.e, d, 64)};
      const Choice s{__shfl_xor(second.v, d, 64), __shfl_xor(second.e, d, 64)};
      const bool better = ranks_before(f, first);
      // the second of both is the loser of the two firsts or the winner's own second
      const Choice lost = better ? first : f, own = better ? s : second;
      first = better ? f : first;
      second = ranks_before(lost, own) ? lost : own;
    }
    const float x1 = L == 1 ? x[1] : __shfl(x[0], (threadIdx.x & 63 & ~(L - 1)) + 1, 64);   // of expert 1
    if (first.e == 0 && x1 != x1) second = {x1, 1};
    if (want_prob) {
      const float top = __shfl(first.v, threadIdx.x & 63 & ~(L - 1), 64);
      double sum = 0.0;
#pragma unroll
      for (int j = 0; j < kRouteValues; ++j) {   // (the first choice's own term is 1 also where it is an infinity)
        const float d = j * L + sub == first.e && x[j] == x[j] ? 0.f : x[j] - top;
        sum += (double)expf(j * L + sub < p.E ? d : -__builtin_inff());
      }
      for (int d = 1; d < L; d <<= 1) sum += __shfl_xor(sum, d, 64);
      if (sub == 0) prob[i] = v2f{(float)(1.0 / sum), (float)((double)expf(second.v - first.v) / sum)};
    }
    if (sub == 0) pair[i] = (unsigned)first.e | (unsigned)second.e << 16;
  }
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
  } else {
    for (int t0 = 0; t0 < p.T; t0 += kRouteBlock) {
      const int n = p.T - t0 < kRouteBlock ? p.T - t0 : kRouteBlock;
      choose_block(p, t0, n, p.row_weight != nullptr && p.chunks == 1, pair, prob);
      __syncthreads();
      if (tid < n) {
        const unsigned c = pair[tid];
        atomicAdd(&total[c & 0xFFFF], 1);
        atomicAdd(&total[c >> 16], 1);
        if (t0 + tid < t_begin) {
          atomicAdd(&before[c & 0xFFFF], 1);
          atomicAdd(&before[c >> 16], 1);
        }
      }
      __syncthreads();
    }
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
    const int n = t_end - t0 < kRouteBlock ? t_end - t0 : kRouteBlock;
    if constexpr (!CHOSEN) {
      if (p.chunks > 1 || p.T > kRouteBlock) {   // (else pair[] and prob[] still hold this block)
        __syncthreads();
        choose_block(p, t0, n, p.row_weight != nullptr, pair, prob);
      }
    }
    for (int i = tid; i < kRouteBlock / 64 * kRouteMaxE; i += kRouteThreads) of_wave[i / kRouteMaxE][i % kRouteMaxE] = 0;
    __syncthreads();
    int expert[2] = {0, 0}, rank[2] = {0, 0};
    v2f weight = {0.f, 0.f};
    const bool on = tid < n;
    if (tid < kRouteBlock) {   // whole waves
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
    }
    __syncthreads();
    if (on) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        int pos = next[expert[k]] + rank[k];
        for (int ww = 0; ww < w; ++ww) pos += of_wave[ww][expert[k]];
        p.token_of_row[pos] = t0 + tid;
        if (p.row_weight) p.row_weight[pos] = weight[k];
        if (p.rows_of_token) p.rows_of_token[2 * (size_t)(t0 + tid) + k] = pos;
      }
    }
    __syncthreads();
    if (tid < kRouteMaxE)
      for (int ww = 0; ww < kRouteBlock / 64; ++ww) next[tid] += of_wave[ww][tid];
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
  if (r.chunks > 1) {   // every workgroup goes through all tokens: more than a few of them only repeat that work
    const int parts = r.chunks < 8 ? r.chunks : 8;
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
