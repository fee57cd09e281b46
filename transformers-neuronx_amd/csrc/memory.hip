// The matrix memory (mLSTM cell): a state S [n, v] a head that is carried from token to token,
//     m' = max(f + m, i),  S' = exp(f + m - m') S + exp(i - m') k val^T,  nrm' likewise with k alone,
//     o = S'^T q / (max(|nrm' . q|, exp(-m')) + 1e-6),
// with i = cap tanh(x_i / cap) and f = logsigmoid(cap tanh(x_f / cap)) from a head's two pre-activations.
// Everything is float32. The state lies in two places by the parity of the position: the token at position p
// reads place (p - 1) & 1 (nothing at p = 0) and writes place p & 1, so a step of single tokens that is run
// twice reads the same both times.
#include <type_traits>

#include "common.h"

TNX_DEFINE_ERROR_API

namespace {

struct CellArgs {
  const float* proj;      // [T, ld]: q [H n] | k [H n] | val [H v] | gate [H v] | x_i [H] | x_f [H]
  int ld;
  const int* run_start;   // [R + 1]
  const int* cached;      // [R]
  const int* slots;       // [R]
  float* memory;          // [slots, 2, H, v, n]
  float* normalizer;      // [slots, 2, H, n]
  float* peak;            // [slots, 2, H]
  float* out;             // [T, H v], before the norm
  int heads, n, v, tokens;
  int chunk_from;         // runs of so many tokens go by chunks, shorter ones token by token
  float cap, q_scale;
};

__device__ __forceinline__ float log_sigmoid(float z) {
  // min(z, 0) - log(1 + exp(-|z|)): neither side overflows
  return fminf(z, 0.f) - log1pf(expf(-fabsf(z)));
}

// The recurrence is taken apart. The gates need nothing of S: one block a (request, head), of as many waves as the
// longest run fills, takes a token a lane and joins their maxima (`memory_gates_kernel`), leaves every token's two factors
// exp(f + m - m'), exp(i - m') and the floor exp(-m') of its denominator in memory, carries m on, and sets the normalizer
// the run begins with aside. Long runs then go by chunks of 64 tokens (`memory_weights_kernel`, `memory_chunks_kernel`),
// the others token by token. The blocks that hold
// S (there `memory_cell_kernel`, 16 columns each) each carry the normalizer along as one more column, so that between
// one token and the next there is nothing but multiply-adds and sums within 16 lanes, and no block reads state
// that another writes: they read the normalizer from where the first kernel set it aside, and the block of a
// head's first columns alone writes it back.
//
// The state lies with a column's rows side by side (`memory` [slots, 2, H, v, n]): a lane's rows of a column are
// neighbours in memory.
//
// A run goes a chunk of tokens at a time through LDS. A token's queries, keys and values lie far from the next
// token's (a row of all heads' projections apart), so what counts is how many loads are under way: every thread
// loads 16 bytes at a time into registers, the next chunk's while this chunk is worked on, and the registers go to
// LDS afterwards. ALIGNED: rows and heads begin at multiples of 16 bytes; otherwise the same with loads of one
// element.

template <bool ALIGNED>
__device__ __forceinline__ f32x4 load4(const float* p, int valid) {      // the first `valid` of four elements, zeros behind
  f32x4 r = {0.f, 0.f, 0.f, 0.f};
  if (valid <= 0) return r;
  if (ALIGNED) return *(const f32x4*)p;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (e < valid) r[e] = p[e];
  return r;
}

// grid: requests * heads blocks of W waves; W 64 tokens a round, a token a lane. The running maximum is a chain
// m' = max(f + m, i) whose steps join: two neighbouring spans (F, I), m -> max(F + m, I), make one of
// (F1 + F2, max(I1 + F2, I2)). A wave joins its lanes' steps in six rounds, the waves before it hand it their spans, and
// every token's m is known at once. (Which m the state is scaled by is free as long as a token's factors name the same m
// on both sides; the joined one differs from the chain's by roundings only.) 2,048 tokens, 32 heads: 102 us with a chain of
// one lane over 64 tokens a round, 10 us so.
template <int W>
__global__ void __launch_bounds__(64 * W) memory_gates_kernel(CellArgs a, float* __restrict__ keeps, float* __restrict__ takes,
                                                              float* __restrict__ floors, float* __restrict__ aside) {
  __shared__ float spans[2][W][2];
  const int r = blockIdx.x / a.heads, head = blockIdx.x - r * a.heads;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int start = a.run_start[r], count = a.run_start[r + 1] - start;
  const int have = a.cached[r], slot = a.slots[r];
  const int hn = a.heads * a.n, hv = a.heads * a.v;
  if (count <= 0) return;
  const int from = (have - 1) & 1, to = (have + count - 1) & 1;
  const size_t head_at = (size_t)slot * 2 * a.heads + head;
  {
    const float* np_ = a.normalizer + (head_at + (size_t)from * a.heads) * a.n;
    float* out = aside + (size_t)blockIdx.x * a.n;
    for (int d = threadIdx.x; d < a.n; d += 64 * W) out[d] = have > 0 ? np_[d] : 0.f;
  }
  float m = have > 0 ? a.peak[head_at + (size_t)from * a.heads] : 0.f;
  int turn = 0;
  for (int t0 = 0; t0 < count; t0 += 64 * W, turn ^= 1) {
    const int t = t0 + threadIdx.x;
    float gi = -INFINITY, gf = 0.f;               // (behind the run's end: a step that changes nothing)
    if (t < count) {
      const float* row = a.proj + (size_t)(start + t) * a.ld + 2 * hn + 2 * hv;
      gi = a.cap * tanhf(row[head] / a.cap);
      gf = log_sigmoid(a.cap * tanhf(row[a.heads + head] / a.cap));
    }
    float F = gf, I = gi;
#pragma unroll
    for (int off = 1; off < 64; off *= 2) {
      const float F0 = __shfl_up(F, off), I0 = __shfl_up(I, off);
      if (lane >= off) I = fmaxf(I0 + F, I), F = F0 + F;
    }
    float next = m;
    if (W > 1) {
      if (lane == 63) spans[turn][wave][0] = F, spans[turn][wave][1] = I;
      __syncthreads();                            // (two places in turn: the next round writes the other)
#pragma unroll
      for (int w = 0; w < W; ++w) {
        if (w == wave) m = next;
        next = fmaxf(spans[turn][w][0] + next, spans[turn][w][1]);
      }
    }
    const float after = fmaxf(F + m, I);
    float before = __shfl_up(after, 1);
    if (lane == 0) before = m;
    if (t < count) {
      const size_t at = (size_t)head * a.tokens + start + t;
      keeps[at] = expf(gf + before - after);
      takes[at] = expf(gi - after);
      floors[at] = expf(-after);
    }
    m = W > 1 ? next : __shfl(after, 63);
  }
  if (threadIdx.x == 0) a.peak[head_at + (size_t)to * a.heads] = m;
}

// ---------------------------------------------------------------- runs by chunks
// Within a chunk of 64 tokens the recurrence is a sum, on the float32 matrix instructions: with P_t the product of the
// chunk's keeps up to token t and D_tj that of the keeps behind token j up to t, times token j's take,
//     S_t^T q_t = P_t S_0^T q_t + sum_{j <= t} (q_t . k_j) D_tj val_j,      S_64 = P_63 S_0 + sum_j D_63,j k_j val_j^T,
// and the same with 1 for val_j for the normalizer. The products of keeps are made token by token, as the walk makes them:
// nothing is divided and no logarithms are subtracted. `memory_weights_kernel` makes (q_t . k_j) D_tj, P_t and D_63,j for all
// chunks side by side; `memory_chunks_kernel` goes through a run's chunks with 16 columns of S a block. The walk is a chain
// of a few multiply-adds and four lane exchanges a token, whatever the matrix units could do. 2,048 tokens, 32 heads of 64
// rows and 128 columns: 399 us by the walk, 124 us by chunks: 19 for the weights and 105 for the chunks (3.3 us each, of
// which the matrix instructions take 0.65: one block of four waves a unit, which waits for its operands). Off from 64 bits
// over 24 draws of 210 to 2,048 tokens, on average: 6.3e-7 of the result by the walk, 4.0e-7 by chunks.
typedef float f32x4v __attribute__((ext_vector_type(4)));

// Chunk `b` of all chunks of 64 tokens of the runs that go by chunks: its run and its first token in it; false: there are fewer.
__device__ __forceinline__ bool find_chunk(const CellArgs& a, int requests, int b, int* run, int* first) {
  for (int r = 0; r < requests; ++r) {
    const int count = a.run_start[r + 1] - a.run_start[r], chunks = count >= a.chunk_from ? (count + 63) >> 6 : 0;
    if (b < chunks) {
      *run = r, *first = 64 * b;
      return true;
    }
    b -= chunks;
  }
  return false;
}

// grid: (chunks, heads), four waves. Wave w makes rows 16 w to 16 w + 15 of the chunk's [64, 64] weights: its 16 queries
// against the keys up to its last row. The factors D: lane j carries token j's through the tokens, a multiplication each.
// weights [H, T, 64], prefix and last [H, T]. NT: 16 NT rows of S hold n.
template <int NT, bool ALIGNED>
__global__ void __launch_bounds__(256) memory_weights_kernel(CellArgs a, int requests, const float* __restrict__ keeps,
                                                             const float* __restrict__ takes, float* __restrict__ weights,
                                                             float* __restrict__ prefix, float* __restrict__ last) {
  constexpr int KD = 4 * NT;                        // elements of a query that a quarter of the lanes holds
  __shared__ float decays[4][16][68];
  int r, c0;
  if (!find_chunk(a, requests, blockIdx.x, &r, &c0)) return;
  const int head = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
  const int start = a.run_start[r] + c0, len = min(64, a.run_start[r + 1] - start);
  const size_t at = (size_t)head * a.tokens + start;
  const int hn = a.heads * a.n;
  const float keep = lane < len ? keeps[at + lane] : 1.f, take = lane < len ? takes[at + lane] : 0.f;
  const float* queries = a.proj + (size_t)start * a.ld + head * a.n + g * KD;
  f32x4v acc[4] = {};
  if (16 * wave < len) {
    f32x4 q[NT];
#pragma unroll
    for (int s = 0; s < NT; ++s)
      q[s] = load4<ALIGNED>(queries + (size_t)min(16 * wave + li, len - 1) * a.ld + 4 * s, a.n - g * KD - 4 * s);
#pragma unroll
    for (int jb = 0; jb < 4; ++jb)
      if (jb <= wave) {
        f32x4 k[NT];
#pragma unroll
        for (int s = 0; s < NT; ++s)
          k[s] = load4<ALIGNED>(queries + hn + (size_t)min(16 * jb + li, len - 1) * a.ld + 4 * s, a.n - g * KD - 4 * s);
#pragma unroll
        for (int s = 0; s < KD; ++s) acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[s / 4][s % 4], k[s / 4][s % 4], acc[jb], 0, 0, 0);
      }
  }
  float D = 0.f, P = 1.f;
  for (int tb = 0; tb <= wave; ++tb) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = 16 * tb + i;
      const float k = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(keep), t));
      D = lane == t ? take : D * k;
      P = lane >= t ? P * k : P;
      if (tb == wave) decays[wave][i][lane] = D;
    }
  }
  if (wave == 3 && lane < len) prefix[at + lane] = P, last[at + lane] = D;
  __syncthreads();
#pragma unroll
  for (int jb = 0; jb < 4; ++jb)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 4 * g + e, t = 16 * wave + i, j = 16 * jb + li;
      if (t < len) weights[(at + t) * 64 + j] = j <= t ? acc[jb][e] * a.q_scale * decays[wave][i][j] : 0.f;
    }
}

// grid: requests * heads * column blocks of 16, four waves. In a chunk wave w makes the outputs of tokens 16 w to 16 w + 15
// and carries rows 16 (w + 4 u) on of S; S as the chunk begins goes round through LDS, in two places in turn, so that a chunk
// has one barrier. Every other operand comes straight from memory in the matrix instruction's own order (a quarter of the
// lanes takes a contiguous quarter of the summed index), a chunk ahead.
template <int NT, bool ALIGNED>
__global__ void __launch_bounds__(256, NT == 4 ? 2 : 1) memory_chunks_kernel(CellArgs a, const float* __restrict__ weights,
                                                            const float* __restrict__ prefix, const float* __restrict__ last,
                                                            const float* __restrict__ floors, const float* __restrict__ aside,
                                                            int column_blocks) {
  constexpr int KD = 4 * NT, NU = NT / 4;
  __shared__ float begins[2][16 * NT * 16 + 64];          // S [row][column]; 16 places more after every quarter of the rows
  __shared__ __attribute__((aligned(16))) float norms[2][16 * NT];
  // A head's queries, keys and weights are read by all its column blocks: eight heads at a time, one an XCD, so that they
  // come into one L2 once. (Blocks go round the XCDs in their order; heads beyond the last eight take theirs as they come.)
  const int heads_by_xcd = gridDim.x / column_blocks & ~7, y = blockIdx.x >> 3;
  const bool by_xcd = blockIdx.x < heads_by_xcd * column_blocks;
  const int cb = (by_xcd ? y : blockIdx.x) % column_blocks;
  const int rh = by_xcd ? 8 * (y / column_blocks) + (blockIdx.x & 7) : blockIdx.x / column_blocks;
  const int r = rh / a.heads, head = rh - r * a.heads;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
  const int start = a.run_start[r], count = a.run_start[r + 1] - start;
  const int have = a.cached[r], slot = a.slots[r];
  const int hn = a.heads * a.n, hv = a.heads * a.v;
  if (count < a.chunk_from) return;
  const int col = 16 * cb + li;
  const bool col_ok = col < a.v;
  const int from = (have - 1) & 1, to = (have + count - 1) & 1;
  const size_t head_at = (size_t)slot * 2 * a.heads + head;        // + place * heads
  f32x4v S[NU];
  float nrm[NU];                                                   // row 16 (wave + 4 u) + li, the same in all quarters
  {
    const float* Sp = a.memory + ((head_at + (size_t)from * a.heads) * a.v + (col_ok ? col : 0)) * a.n;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int d0 = 16 * (wave + 4 * u);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = d0 + 4 * g + e;
        S[u][e] = (have > 0 && d < a.n && col_ok) ? Sp[d] : 0.f;
      }
      nrm[u] = d0 + li < a.n ? aside[(size_t)rh * a.n + d0 + li] : 0.f;
    }
  }
  f32x4 q[NT], w[4];
  float k[NU][16], v[16], ends[16], mine, floor_, keep;
  // (every load is made, of the run's last token's row behind its end and of the first column or row of S beyond the last
  // one: what they bring is multiplied by a weight of zero or belongs to places that are not stored. A whole chunk's rows
  // are a fixed distance apart.)
  const int vcol = 2 * hn + head * a.v + (col_ok ? col : 0);
  int krow[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int d = 16 * (wave + 4 * u) + li;
    krow[u] = hn + head * a.n + (d < a.n ? d : 0);
  }
  auto fetch_rows = [&](int c0, int len, auto whole) __attribute__((always_inline)) {
    const size_t at = (size_t)head * a.tokens + start + c0;
    const float* rows = a.proj + (size_t)(start + c0) * a.ld;
    const int t = whole ? 16 * wave + li : min(16 * wave + li, len - 1);
#pragma unroll
    for (int s = 0; s < NT; ++s)
      q[s] = load4<ALIGNED>(rows + (size_t)t * a.ld + head * a.n + g * KD + 4 * s, a.n - g * KD - 4 * s);
#pragma unroll
    for (int s = 0; s < 4; ++s) w[s] = *(const f32x4*)(weights + (at + t) * 64 + 16 * g + 4 * s);
    mine = prefix[at + t], floor_ = floors[at + t], keep = prefix[at + len - 1];
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      const int j = whole ? 16 * g + s : min(16 * g + s, len - 1);
      const float* row = whole ? rows + (size_t)s * a.ld + 16 * g * a.ld : rows + (size_t)j * a.ld;
      v[s] = row[vcol];
      ends[s] = last[at + j];
#pragma unroll
      for (int u = 0; u < NU; ++u) k[u][s] = row[krow[u]];
    }
  };
  auto fetch = [&](int c0) __attribute__((always_inline)) {
    const int len = count - c0;
    if (len >= 64)
      fetch_rows(c0, 64, std::true_type());
    else
      fetch_rows(c0, len, std::false_type());
  };
  fetch(0);
  int turn = 0;
  for (int c0 = 0; c0 < count; c0 += 64, turn ^= 1) {
    const int len = min(64, count - c0);
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int d0 = 16 * (wave + 4 * u);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = d0 + 4 * g + e;
        begins[turn][16 * (d + d / KD) + li] = S[u][e];
      }
      if (g == 0) norms[turn][d0 + li] = nrm[u];
    }
    __syncthreads();
    // this chunk's operands, made ready; then the next chunk's are asked for
    f32x4 ww[4];
    float qq[KD], kk[NU][16], vv[16];
    const float scale = a.q_scale * mine, floor_now = floor_, keep_now = keep;
#pragma unroll
    for (int s = 0; s < KD; ++s) qq[s] = q[s / 4][s % 4] * scale;
#pragma unroll
    for (int s = 0; s < 4; ++s) ww[s] = w[s];
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      // (behind the run's end nothing, also of the last token's value: where that is infinite, zero times it is no number)
      vv[s] = 16 * g + s < len ? v[s] : 0.f;
#pragma unroll
      for (int u = 0; u < NU; ++u) kk[u][s] = 16 * g + s < len ? k[u][s] * ends[s] : 0.f;
    }
    if (c0 + 64 < count) fetch(c0 + 64);
    f32x4v acc = {}, more = {};
    float dot = 0.f, probe = 0.f;
#pragma unroll
    for (int s = 0; s < KD; ++s) {
      const int d = g * KD + s;
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(qq[s], begins[turn][16 * (d + g) + li], acc, 0, 0, 0);
      dot += qq[s] * norms[turn][d];
    }
#pragma unroll
    for (int s = 0; s < 16; ++s) probe += vv[s] * 0.f;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      float sum = 0.f;
      S[u] *= keep_now;
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        S[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[u][s], vv[s], S[u], 0, 0, 0);
        sum += kk[u][s];
      }
      sum += __shfl_xor(sum, 16);
      sum += __shfl_xor(sum, 32);
      nrm[u] = keep_now * nrm[u] + sum;
    }
    // A value that is infinite or no number must not reach the tokens before it, whose weight of it is zero: it is left out
    // of the products, and the tokens from it on are no numbers in its column. (The walk adds up a row of S at a time: there
    // an infinite value is an infinity of either sign a row, whose sum is no number either unless a token's products q_d k_d
    // all have one sign, one token in 500 at 10 rows and none to speak of at 16.)
    int spoilt = 64;
    if (__any(probe != 0.f)) {
#pragma unroll
      for (int s = 15; s >= 0; --s)
        if (vv[s] * 0.f != 0.f) vv[s] = 0.f, spoilt = 16 * g + s;
      spoilt = min(spoilt, __shfl_xor(spoilt, 16));
      spoilt = min(spoilt, __shfl_xor(spoilt, 32));
    }
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      more = __builtin_amdgcn_mfma_f32_16x16x4f32(ww[s / 4][s % 4], vv[s], more, 0, 0, 0);
      dot += ww[s / 4][s % 4];
    }
    dot += __shfl_xor(dot, 16);
    dot += __shfl_xor(dot, 32);
    // (the denominator is 1e-6 at least: its reciprocal, right to a unit in the last place, is no subnormal)
    const float below = __builtin_amdgcn_rcpf(fmaxf(fabsf(dot), floor_now) + 1e-6f);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 16 * wave + 4 * g + e;
      const float o = (acc[e] + more[e]) * __shfl(below, 4 * g + e);
      if (t < len && col_ok) a.out[(size_t)(start + c0 + t) * hv + head * a.v + col] = t < spoilt ? o : NAN;
    }
  }
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int d0 = 16 * (wave + 4 * u);
    if (col_ok) {
      float* Sp = a.memory + ((head_at + (size_t)to * a.heads) * a.v + col) * a.n;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (d0 + 4 * g + e < a.n) Sp[d0 + 4 * g + e] = S[u][e];
    }
    if (cb == 0 && g == 0 && d0 + li < a.n)                        // the normalizer, once a head
      a.normalizer[(head_at + (size_t)to * a.heads) * a.n + d0 + li] = nrm[u];
  }
}

// ---------------------------------------------------------------- runs token by token
// grid: requests * heads * column blocks; a block is four waves and 16 columns of S. In a wave the 16 lanes of a
// row of lanes share a column (column 16 b + 4 w + lane / 16): lane % 16 holds its rows NR (lane % 16) + j, j < NR,
// and the same rows of the normalizer; a column's sum over the rows is a sum over the 16 lanes of a row of lanes.
template <int NR, bool ALIGNED>
__global__ void __launch_bounds__(256) memory_cell_kernel(CellArgs a, const float* __restrict__ keeps,
                                                          const float* __restrict__ takes,
                                                          const float* __restrict__ floors,
                                                          const float* __restrict__ aside, int column_blocks) {
  constexpr int CH = NR == 16 ? 16 : 32;                  // tokens a chunk
  constexpr int np = 16 * NR;                             // a token's queries (and keys) in LDS, zeros behind n
  constexpr int PT = np / 4;                              // 16-byte pieces of a token's queries
  constexpr int QN = (CH * PT + 255) / 256;               // pieces of queries (and keys) a thread and chunk
  __shared__ __attribute__((aligned(16))) float qs[CH * np];      // queries, scaled
  __shared__ __attribute__((aligned(16))) float ks[CH * np];      // keys times exp(i - m')
  __shared__ __attribute__((aligned(16))) float vs[CH * 16];
  __shared__ float kp[CH], fl[CH];                        // exp(f + m - m'), exp(-m')
  const int cb = blockIdx.x % column_blocks, rh = blockIdx.x / column_blocks;
  const int r = rh / a.heads, head = rh - r * a.heads;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int grp = lane & 15;
  const int start = a.run_start[r], count = a.run_start[r + 1] - start;
  const int have = a.cached[r], slot = a.slots[r];
  const int hn = a.heads * a.n, hv = a.heads * a.v;
  if (count <= 0 || count >= a.chunk_from) return;
  const int col = 16 * cb + 4 * wave + (lane >> 4);
  const bool col_ok = col < a.v;
  float S[NR], nrm[NR];
  const int from = (have - 1) & 1, to = (have + count - 1) & 1;
  const size_t head_at = (size_t)slot * 2 * a.heads + head;        // + place * heads
  {
    const float* Sp = a.memory + ((head_at + (size_t)from * a.heads) * a.v + (col_ok ? col : 0)) * a.n;
    const float* np_ = aside + (size_t)rh * a.n;
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      const int d = grp * NR + j;
      S[j] = (have > 0 && d < a.n && col_ok) ? Sp[d] : 0.f;
      nrm[j] = d < a.n ? np_[d] : 0.f;
    }
  }
  const size_t run_at = (size_t)head * a.tokens + start;
  const float *my_keeps = keeps + run_at, *my_takes = takes + run_at, *my_floors = floors + run_at;
  f32x4 rq[QN], rk[QN], rv = {0.f, 0.f, 0.f, 0.f};
  float rt[QN], rkeep = 1.f, rfl = 0.f;
  auto fetch = [&](int t0) {
    const int len = min(CH, count - t0);
#pragma unroll
    for (int u = 0; u < QN; ++u) {
      const int f = threadIdx.x + 256 * u, t = f / PT, d = 4 * (f - t * PT);
      const bool in = f < CH * PT && t < len;
      const float* row = a.proj + (size_t)(start + t0 + (in ? t : 0)) * a.ld + head * a.n + d;
      rq[u] = load4<ALIGNED>(row, in ? a.n - d : 0);
      rk[u] = load4<ALIGNED>(row + hn, in ? a.n - d : 0);
      rt[u] = in ? my_takes[t0 + t] : 0.f;
    }
    if (threadIdx.x < CH * 4) {                            // a token's 16 values: four pieces
      const int t = threadIdx.x >> 2, c = 16 * cb + 4 * (threadIdx.x & 3);
      const bool in = t < len;
      rv = load4<ALIGNED>(a.proj + (size_t)(start + t0 + (in ? t : 0)) * a.ld + 2 * hn + head * a.v + c, in ? a.v - c : 0);
    }
    if (threadIdx.x < CH) {
      const bool in = threadIdx.x < len;
      rkeep = in ? my_keeps[t0 + threadIdx.x] : 1.f;
      rfl = in ? my_floors[t0 + threadIdx.x] : 1.f;
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int u = 0; u < QN; ++u) {
      const int f = threadIdx.x + 256 * u;                // piece f of the chunk: token f / PT, elements 4 (f % PT) on
      if (f < CH * PT) {
        *(f32x4*)(qs + 4 * f) = rq[u] * a.q_scale;
        *(f32x4*)(ks + 4 * f) = rk[u] * rt[u];
      }
    }
    if (threadIdx.x < CH * 4) *(f32x4*)(vs + 4 * threadIdx.x) = rv;
    if (threadIdx.x < CH) kp[threadIdx.x] = rkeep, fl[threadIdx.x] = rfl;
  };
  fetch(0);
  stash();
  __syncthreads();
  for (int t0 = 0; t0 < count; t0 += CH) {
    const int len = min(CH, count - t0);
    const bool more = t0 + CH < count;
    if (more) fetch(t0 + CH);                             // under way while this chunk is worked on
    // a token's operands are read from LDS while the token before it is worked on
    float q_n[NR], k_n[NR], val_n, keep_n, fl_n;
    auto read = [&](int t) {
      const float* q = qs + t * np + grp * NR;
      const float* k = ks + t * np + grp * NR;
#pragma unroll
      for (int j = 0; j < NR; ++j) q_n[j] = q[j], k_n[j] = k[j];
      val_n = vs[t * 16 + 4 * wave + (lane >> 4)];
      keep_n = kp[t];
      fl_n = fl[t];
    };
    auto token = [&](int t, bool last) {
      float q[NR], k[NR];
#pragma unroll
      for (int j = 0; j < NR; ++j) q[j] = q_n[j], k[j] = k_n[j];
      const float val = val_n, keep = keep_n, floor_ = fl_n;
      if (!last) read(t + 1);
      float top = 0.f, dot = 0.f;
#pragma unroll
      for (int j = 0; j < NR; ++j) {
        S[j] = keep * S[j] + k[j] * val;
        nrm[j] = keep * nrm[j] + k[j];
        top += S[j] * q[j];
        dot += nrm[j] * q[j];
      }
      // sums over the 16 lanes of a row of lanes
      top += lane_dpp<TNX_DPP_XOR1>(top), dot += lane_dpp<TNX_DPP_XOR1>(dot);
      top += lane_dpp<TNX_DPP_XOR2>(top), dot += lane_dpp<TNX_DPP_XOR2>(dot);
      top += lane_dpp<TNX_DPP_HALF_MIRROR>(top), dot += lane_dpp<TNX_DPP_HALF_MIRROR>(dot);
      top += lane_dpp<TNX_DPP_MIRROR>(top), dot += lane_dpp<TNX_DPP_MIRROR>(dot);
      // (the denominator is 1e-6 at least: its reciprocal, right to a unit in the last place, is no subnormal)
      const float o = top * __builtin_amdgcn_rcpf(fmaxf(fabsf(dot), floor_) + 1e-6f);
      if (grp == 0 && col_ok) a.out[(size_t)(start + t0 + t) * hv + head * a.v + col] = o;
    };
    read(0);
    if (len == CH) {        // a whole chunk: a count the compiler knows
#pragma unroll 4
      for (int t = 0; t < CH; ++t) token(t, t == CH - 1);
    } else {
      for (int t = 0; t < len; ++t) token(t, t == len - 1);
    }
    __syncthreads();        // before the next chunk takes the place of what this one read
    if (more) {
      stash();
      __syncthreads();
    }
  }
  if (col_ok) {
    float* Sp = a.memory + ((head_at + (size_t)to * a.heads) * a.v + col) * a.n;
#pragma unroll
    for (int j = 0; j < NR; ++j)
      if (grp * NR + j < a.n) Sp[grp * NR + j] = S[j];
  }
  if (cb == 0 && wave == 0 && lane < 16) {                 // the normalizer, once a head
    float* np_ = a.normalizer + (head_at + (size_t)to * a.heads) * a.n;
#pragma unroll
    for (int j = 0; j < NR; ++j)
      if (grp * NR + j < a.n) np_[grp * NR + j] = nrm[j];
  }
}

// What follows the cell up to the output projection: each head's o at unit root mean square, weighted, times
// sigmoid(gate); a wave a (token, head).
template <typename T>
__global__ void __launch_bounds__(256) memory_output_kernel(const float* __restrict__ o, const float* __restrict__ proj,
                                                            int ld, int gate_at, const float* __restrict__ weight,
                                                            float eps, T* __restrict__ out, int pairs, int heads, int v) {
  const int pair = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (pair >= pairs) return;
  const int t = pair / heads, head = pair - t * heads;
  const float* mine = o + (size_t)t * heads * v + head * v;
  float s = 0.f;
  for (int i = lane; i < v; i += 64) s += mine[i] * mine[i];
  s = wave_sum(s);
  const float r = 1.f / sqrtf(s / (float)v + eps);
  const float* gate = proj + (size_t)t * ld + gate_at + head * v;
  for (int i = lane; i < v; i += 64) {
    const float g = 1.f / (1.f + expf(-gate[i]));
    out[(size_t)t * heads * v + head * v + i] = from_f32<T>(mine[i] * r * weight[head * v + i] * g);
  }
}

template <int NR>
void launch_cell(const CellArgs& a, const float* keeps, const float* takes, const float* floors, const float* aside,
                 int requests, bool aligned, hipStream_t stream) {
  const int column_blocks = (a.v + 15) / 16;
  const dim3 grid(requests * a.heads * column_blocks);
  if (aligned)
    memory_cell_kernel<NR, true><<<grid, 256, 0, stream>>>(a, keeps, takes, floors, aside, column_blocks);
  else
    memory_cell_kernel<NR, false><<<grid, 256, 0, stream>>>(a, keeps, takes, floors, aside, column_blocks);
}

template <int NT>
void launch_chunks(const CellArgs& a, const float* keeps, const float* takes, const float* floors, const float* aside,
                   float* work, int requests, bool aligned, hipStream_t stream) {
  const size_t th = (size_t)a.tokens * a.heads;
  float *weights = work, *prefix = work + 64 * th, *last = work + 65 * th;
  const dim3 chunks(a.tokens / 64 + requests, a.heads);
  const int column_blocks = (a.v + 15) / 16;
  const dim3 grid(requests * a.heads * column_blocks);
  if (aligned) {
    memory_weights_kernel<NT, true><<<chunks, 256, 0, stream>>>(a, requests, keeps, takes, weights, prefix, last);
    memory_chunks_kernel<NT, true><<<grid, 256, 0, stream>>>(a, weights, prefix, last, floors, aside, column_blocks);
  } else {
    memory_weights_kernel<NT, false><<<chunks, 256, 0, stream>>>(a, requests, keeps, takes, weights, prefix, last);
    memory_chunks_kernel<NT, false><<<grid, 256, 0, stream>>>(a, weights, prefix, last, floors, aside, column_blocks);
  }
}

}  // namespace

// `longest`, `shortest`: the tokens of the step's longest and shortest run. Runs of `chunk_from` tokens go by chunks
// (query/key heads of up to 128 elements; `chunk_work`: 66 floats a token and head, 16 bytes aligned), shorter ones, and
// all where `chunk_work` is null, token by token.
extern "C" int tnx_matrix_memory(const float* proj, int ld, const int* run_start, const int* cached, const int* slots,
                                 float* memory, float* normalizer, float* peak, int num_slots, float* raw, float* gates,
                                 int longest, int shortest, int chunk_from, float* chunk_work,
                                 const float* weight, float eps, void* out, int dtype, int tokens, int requests, int heads,
                                 int n, int v, float cap, hipStream_t stream) {
  TNX_REQUIRE(tokens >= 0 && requests >= 0 && heads > 0 && n > 0 && v > 0, "matrix_memory: bad sizes");
  TNX_REQUIRE(n <= 256, "matrix_memory: query/key heads of up to 256 elements, got %d", n);
  TNX_REQUIRE(ld >= 2 * heads * n + 2 * heads * v + 2 * heads, "matrix_memory: rows of %d elements, %d needed", ld,
              2 * heads * n + 2 * heads * v + 2 * heads);
  TNX_REQUIRE(cap > 0.f, "matrix_memory: the gates' cap must be positive");
  TNX_REQUIRE(dtype == TNX_F32 || dtype == TNX_BF16, "matrix_memory: dtype %d", dtype);
  if (tokens == 0 || requests == 0) return 0;
  CellArgs a{proj, ld, run_start, cached, slots, memory, normalizer, peak, raw, heads, n, v, tokens,
             chunk_work != nullptr ? (chunk_from > 1 ? chunk_from : 1) : 0x7fffffff, cap, 1.f / sqrtf((float)n)};
  TNX_REQUIRE(chunk_work == nullptr || (n <= 128 && heads <= 65535 && (uintptr_t)chunk_work % 16 == 0),
              "matrix_memory: by chunks: query/key heads of up to 128 elements, room at a multiple of 16 bytes");
  float* keeps = gates;                             // [H, T] each
  float* takes = gates + (size_t)tokens * heads;
  float* floors = gates + 2 * (size_t)tokens * heads;
  float* aside = gates + 3 * (size_t)tokens * heads;      // [R, H, n]: the normalizers the runs begin with
  // rows and heads that begin at multiples of 16 bytes are loaded 16 bytes at a time
  const bool aligned = n % 4 == 0 && v % 4 == 0 && ld % 4 == 0 && (uintptr_t)proj % 16 == 0;
  // as many waves as the longest run fills
  if (longest <= 64)
    memory_gates_kernel<1><<<requests * heads, 64, 0, stream>>>(a, keeps, takes, floors, aside);
  else if (longest <= 256)
    memory_gates_kernel<4><<<requests * heads, 256, 0, stream>>>(a, keeps, takes, floors, aside);
  else
    memory_gates_kernel<16><<<requests * heads, 1024, 0, stream>>>(a, keeps, takes, floors, aside);
  TNX_CHECK_LAUNCH("matrix_memory gates");
  const int rows16 = (n + 15) / 16;
  if (longest >= a.chunk_from) {
    if (rows16 <= 4)
      launch_chunks<4>(a, keeps, takes, floors, aside, chunk_work, requests, aligned, stream);
    else
      launch_chunks<8>(a, keeps, takes, floors, aside, chunk_work, requests, aligned, stream);
  }
  if (shortest < a.chunk_from) {
    if (rows16 <= 2)
      launch_cell<2>(a, keeps, takes, floors, aside, requests, aligned, stream);
    else if (rows16 <= 4)
      launch_cell<4>(a, keeps, takes, floors, aside, requests, aligned, stream);
    else if (rows16 <= 8)
      launch_cell<8>(a, keeps, takes, floors, aside, requests, aligned, stream);
    else
      launch_cell<16>(a, keeps, takes, floors, aside, requests, aligned, stream);
  }
  TNX_CHECK_LAUNCH("matrix_memory");
  const int pairs = tokens * heads;
  const int gate_at = 2 * heads * n + heads * v;
  if (dtype == TNX_F32)
    memory_output_kernel<float><<<(pairs + 3) / 4, 256, 0, stream>>>(raw, proj, ld, gate_at, weight, eps, (float*)out,
                                                                      pairs, heads, v);
  else
    memory_output_kernel<bf16_t><<<(pairs + 3) / 4, 256, 0, stream>>>(raw, proj, ld, gate_at, weight, eps, (bf16_t*)out,
                                                                       pairs, heads, v);
  TNX_CHECK_LAUNCH("matrix_memory output");
  return 0;
}
