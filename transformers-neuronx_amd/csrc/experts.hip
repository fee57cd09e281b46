// A mixture of experts: the router's choice, the step's (token, choice) pairs put in the order of their
// experts, and the two products of every expert over its own pairs,
//     inner = act(w g) * (w u)  with [g | u] = W_gate_up[e] h      (the weight w on the expert's input; on its
//     y = W_down[e] inner                                           output it multiplies y instead)
// or, for experts without a gate, inner = act(W_up[e] h),
// summed over a token's choices onto the residual in float32. Nothing is read back by the host: the launches are
// sized by the most tiles the pairs can make, and a block that finds no tile ends at once.
#include "tiles.h"

TNX_DEFINE_ERROR_API

namespace {

// ---------------------------------------------------------------- the router's choice
// A wave a token: `top` rounds of the largest logit (the lower number where two are equal), whose score sigmoid(z)
// or softmax(z) is the weight. The ranking is by the logits, which both scores grow with: two large logits that
// float32 still tells apart can have scores that it does not. With `correction` (a number an expert) the ranking is
// by score + correction, and the weight is the score without it; `scale` multiplies every weight. With `keep` < `groups`
// the experts form that many equal groups of neighbours, a group ranks by its best expert, and only experts of the `keep`
// best groups (the lower number where two are equal) take part.
constexpr int MAX_GROUPS = 256;
struct RouteArgs {
  int tokens, experts, top, softmax, renormalize;
  int* chosen;
  float* weights;
  const float* correction;
  float scale;
  int groups, keep;
};

// Token t's choice from its logits `row` (global memory or LDS), by one wave; `best`, `kept`: the wave's room for the groups.
__device__ __forceinline__ void route_token(const RouteArgs& a, const float* row, int t, float* best, unsigned char* kept) {
  const int lane = threadIdx.x & 63, experts = a.experts, top = a.top, softmax = a.softmax, groups = a.groups, keep = a.keep;
  int* chosen = a.chosen;
  float* weights = a.weights;
  const float *correction = a.correction, scale = a.scale;
  float peak = -INFINITY, total = 1.f;
  if (softmax) {
    for (int e = lane; e < experts; e += 64) peak = fmaxf(peak, row[e]);
    peak = wave_max(peak);
    float s = 0.f;
    for (int e = lane; e < experts; e += 64) s += expf(row[e] - peak);
    total = wave_sum(s);
  }
  auto score = [&](float z) { return softmax ? expf(z - peak) / total : 1.f / (1.f + expf(-z)); };
  auto plain_rank = [&](int e) { return correction ? score(row[e]) + correction[e] : row[e]; };
  const int per = experts / groups;
  const bool grouped = keep < groups;
  if (grouped) {      // (a wave's own rows of LDS; a wave's LDS operations keep their order)
    for (int g = 0; g < groups; ++g) {
      float b = -INFINITY;
      for (int e = lane; e < per; e += 64) b = fmaxf(b, plain_rank(g * per + e));
      b = wave_max(b);
      if (lane == 0) best[g] = b, kept[g] = 0;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int c = 0; c < keep; ++c) {
      float b = -INFINITY;
      int at = groups;
      for (int g = lane; g < groups; g += 64)
        if (!kept[g] && (best[g] > b || at == groups)) b = best[g], at = g;
      const float high = wave_max(b);
      const int first = -(int)wave_max((float)-((b == high && at < groups) ? at : groups));
      if (lane == 0 && first < groups) kept[first] = 1;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
  auto rank = [&](int e) { return !grouped || kept[e / per] ? plain_rank(e) : -INFINITY; };
  float sum = 0.f;
  unsigned long long taken = 0;        // bit i: expert lane + 64 i is chosen already (a lane's own experts)
  for (int c = 0; c < top; ++c) {
    float best = -INFINITY;
    int at = experts;
    for (int e = lane, i = 0; e < experts; e += 64, ++i) {
      const float z = rank(e);
      if (!((taken >> i) & 1) && (z > best || at == experts)) best = z, at = e;   // ascending e: the lower number stays where two are equal
    }
    const float high = wave_max(best);
    const int first = -(int)wave_max((float)-((best == high && at < experts) ? at : experts));
    if ((first & 63) == lane) taken |= 1ull << (first >> 6);
    const float s = correction ? score(row[first]) : score(high);
    if (lane == 0) {
      chosen[(size_t)t * top + c] = first;
      weights[(size_t)t * top + c] = a.renormalize ? 0.f : s * scale;
    }
    sum += s;
  }
  if (a.renormalize) {
    // the same rounds again, now that the sum is known: each weight is written once
    taken = 0;
    for (int c = 0; c < top; ++c) {
      float best = -INFINITY;
      int at = experts;
      for (int e = lane, i = 0; e < experts; e += 64, ++i) {
        const float z = rank(e);
        if (!((taken >> i) & 1) && (z > best || at == experts)) best = z, at = e;
      }
      const float high = wave_max(best);
      const int first = -(int)wave_max((float)-((best == high && at < experts) ? at : experts));
      if ((first & 63) == lane) taken |= 1ull << (first >> 6);
      if (lane == 0) weights[(size_t)t * top + c] = (correction ? score(row[first]) : score(high)) / sum * scale;
    }
  }
}

__global__ void __launch_bounds__(256) route_kernel(const float* __restrict__ z, int ld, RouteArgs a) {
  __shared__ float best_of[4][MAX_GROUPS];        // a wave's groups: the best rank, and whether the group is kept
  __shared__ unsigned char kept_of[4][MAX_GROUPS];
  const int wave = threadIdx.x >> 6, t = blockIdx.x * 4 + wave;
  if (t < a.tokens) route_token(a, z + (size_t)t * ld, t, best_of[wave], kept_of[wave]);
}

// The router's product and the choice in one launch, a block a token: z = W_r h + bias (bfloat16 operands, exact products,
// float32 sums of 8 to 16 elements a thread, then by tree), eight experts at a time. A launch costs 3 to 5 us here and this work a
// fraction of it: what bounds it is the block's few readings of memory one after the other, and for many tokens the matrix, which every
// block reads from the cache. us, a launch for the product and one for the choice / this: 8 experts, rows of 2,048, 1 token 6.2 / 4.3, 8 tokens 7.4 / 4.6,
// 396 9.6 / 5.2, 2,048 8.2 / 8.4; rows of 4,096, 8 tokens 9.8 / 5.1, 2,048 9.7 / 10.2; 16 of 2,880, 8 tokens 9.8 / 6.8, 396 9.8 / 7.8, 2,048 11.2 / 15.1;
// 32 of 2,048, 8 tokens 7.2 / 9.1.
constexpr int ROUTE_PRODUCT_MOST = 16;     // experts
__global__ void __launch_bounds__(256) route_product_kernel(const bf16_t* __restrict__ h, const bf16_t* __restrict__ w,
                                                            const float* __restrict__ bias, int width, RouteArgs a) {
  __shared__ float parts[4][ROUTE_PRODUCT_MOST], z[ROUTE_PRODUCT_MOST], best[ROUTE_PRODUCT_MOST];
  __shared__ unsigned char kept[ROUTE_PRODUCT_MOST];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bf16_t* row = h + (size_t)t * width;
  for (int e0 = 0; e0 < a.experts; e0 += 8) {
    float sum[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) sum[e] = 0.f;
    for (int k = 8 * tid; k < width; k += 2048) {
      const bf16x8 x = *(const bf16x8*)(row + k);
      bf16x8 v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = *(const bf16x8*)(w + (size_t)min(e0 + e, a.experts - 1) * width + k);
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int i = 0; i < 8; ++i) sum[e] = fmaf((float)x[i], (float)v[e][i], sum[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float s = wave_sum(sum[e]);
      if (lane == 0 && e0 + e < a.experts) parts[wave][e0 + e] = s;
    }
  }
  __syncthreads();
  if (wave) return;
  if (lane < a.experts)
    z[lane] = (parts[0][lane] + parts[1][lane]) + (parts[2][lane] + parts[3][lane]) + (bias ? bias[lane] : 0.f);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  route_token(a, z, t, best, kept);
}

// ---------------------------------------------------------------- pairs in the order of their experts
// One block: counts an expert, where each expert's pairs begin (`first[E + 1]`), and the pairs (t * top + c)
// put there (`order`). The order within an expert changes no result: every pair's row is computed alone.
__global__ void __launch_bounds__(1024) order_kernel(const int* __restrict__ chosen, int pairs, int experts,
                                                     int* __restrict__ first, int* __restrict__ order,
                                                     int* __restrict__ place, int* __restrict__ token, int top,
                                                     const float* __restrict__ weights, float* __restrict__ sorted_weights,
                                                     int2* __restrict__ tiles, int tile_rows, int tile_slots) {
  extern __shared__ int counts[];      // [experts] counts, then [experts] cursors, then (with `tiles`) [experts] first tiles
  __shared__ int tiles_used;
  int* cursor = counts + experts;
  int* tile_at = cursor + experts;
  for (int e = threadIdx.x; e < experts; e += blockDim.x) counts[e] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < pairs; i += blockDim.x) {
    const int e = chosen[i];
    if (e >= 0 && e < experts) atomicAdd(&counts[e], 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int at = 0, used = 0;
    for (int e = 0; e < experts; ++e) {
      first[e] = at;
      cursor[e] = at;
      at += counts[e];
      if (tiles) {
        tile_at[e] = used;
        used += (counts[e] + tile_rows - 1) / tile_rows;
      }
    }
    first[experts] = at;
    tiles_used = used;
  }
  __syncthreads();
  if (tiles) {
    // tile i: an expert and the first of its sorted rows; an expert of -1 where there are fewer tiles than slots
    for (int e = threadIdx.x; e < experts; e += blockDim.x)
      for (int r = 0, i = tile_at[e]; r < counts[e]; r += tile_rows, ++i) tiles[i] = make_int2(e, cursor[e] + r);
    for (int i = tiles_used + threadIdx.x; i < tile_slots; i += blockDim.x) tiles[i] = make_int2(-1, 0);
    if (threadIdx.x == 0) tiles[tile_slots] = make_int2(tiles_used, 0);      // and behind them how many there are
    __syncthreads();                   // the cursors move from here on
  }
  for (int i = threadIdx.x; i < pairs; i += blockDim.x) {
    const int e = chosen[i];
    if (e >= 0 && e < experts) {
      const int at = atomicAdd(&cursor[e], 1);
      order[at] = i;
      if (place) place[i] = at;                       // where the pair's row lies among the sorted ones
      if (token) token[at] = i / top;                 // the token whose row the sorted row reads
      if (sorted_weights) sorted_weights[at] = weights[i];
    }
  }
}

// ---------------------------------------------------------------- an expert's product over its pairs
// out[pair, j] = sum_k A[row(pair), k] W[e][j][k] for the pairs of expert e, a tile of 16 pairs by 64 columns a
// block, float32 sums from tiles staged in LDS. UP_GATED: W holds F gate rows and then F up rows, column j of the
// result is act(w g_j) * (w u_j) and the A row of a pair is its token's (pair / top); UP_PLAIN: W holds F rows, the
// result is act(u_j). DOWN: the A row is the pair's own, and the result goes to `out` (pair rows, float32) or, where a
// token has one choice, straight onto the residual into the token's row.
constexpr int DOWN = 0, UP_GATED = 1, UP_PLAIN = 2;
struct ProductArgs {
  const void* a;            // UP: h [T, K]; DOWN: inner [pairs, K]
  const void* w;            // [E, N(, 2), K]
  const int* first;         // [E + 1]
  const int* order;         // [pairs]
  const float* weights;     // [pairs]
  const float* residual;    // [T, N] or null (DOWN, one choice a token)
  void* out;
  int experts, top, n, k, act, weight_on_input, pairs;
  float limit;              // of the clamped activation
  int direct;               // DOWN: pair rows are the tokens' rows of the result, and take the residual
  const int* chosen;        // [pairs], up to 64 pairs: the blocks find an expert's pairs in it themselves (no `first`, `order`)
};

template <typename T, int KIND>
__global__ void __launch_bounds__(256) expert_product_kernel(ProductArgs p) {
  constexpr bool GATED = KIND == UP_GATED, UP = KIND != DOWN;
  constexpr int TM = 16, TN = 64, TK = 32;
  __shared__ float As[TM][TK + 1];
  __shared__ float Ws[GATED ? 2 : 1][TN][TK + 1];
  __shared__ int rows[TM];
  // which expert and which of its tiles of 16 pairs this block is
  int tile = blockIdx.y, e = 0, begin = 0, end = 0;
  for (; e < p.experts; ++e) {
    begin = p.first[e];
    end = p.first[e + 1];
    const int tiles = (end - begin + TM - 1) / TM;
    if (tile < tiles) break;
    tile -= tiles;
  }
  if (e >= p.experts) return;
  begin += tile * TM;
  const int count = min(TM, end - begin);
  const int col0 = blockIdx.x * TN;
  if (threadIdx.x < TM) rows[threadIdx.x] = threadIdx.x < count ? p.order[begin + threadIdx.x] : -1;
  __syncthreads();
  const T* A = (const T*)p.a;
  const T* W = (const T*)p.w + (size_t)e * (GATED ? 2 : 1) * p.n * p.k;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;        // column, and rows 4 ty .. 4 ty + 3
  float acc[GATED ? 2 : 1][4] = {};
  for (int k0 = 0; k0 < p.k; k0 += TK) {
    // the tile of A: 16 rows of 32, two elements a thread
    for (int i = threadIdx.x; i < TM * TK; i += 256) {
      const int r = i / TK, c = i - r * TK;
      const int pair = rows[r];
      float v = 0.f;
      if (pair >= 0 && k0 + c < p.k) v = to_f32(A[(size_t)(UP ? pair / p.top : pair) * p.k + k0 + c]);
      As[r][c] = v;
    }
    // the tile of W: 64 (or twice 64) rows of 32
    for (int i = threadIdx.x; i < (GATED ? 2 : 1) * TN * TK; i += 256) {
      const int half = i / (TN * TK), j = (i - half * TN * TK) / TK, c = i % TK;
      float v = 0.f;
      if (col0 + j < p.n && k0 + c < p.k) v = to_f32(W[((size_t)half * p.n + col0 + j) * p.k + k0 + c]);
      Ws[half][j][c] = v;
    }
    __syncthreads();
#pragma unroll 8
    for (int c = 0; c < TK; ++c) {
      const float w0 = Ws[0][tx][c];
      const float w1 = GATED ? Ws[GATED ? 1 : 0][tx][c] : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = As[4 * ty + r][c];
        acc[0][r] += x * w0;
        if (GATED) acc[GATED ? 1 : 0][r] += x * w1;
      }
    }
    __syncthreads();
  }
  const int col = col0 + tx;
  if (col >= p.n) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int pair = rows[4 * ty + r];
    if (pair < 0) continue;
    const float w = p.weights[pair];
    if (GATED) {
      float g = acc[0][r], u = acc[GATED ? 1 : 0][r];
      if (p.weight_on_input) g *= w, u *= w;
      with_gate(p.act, p.limit, [&](auto gate) { ((T*)p.out)[(size_t)pair * p.n + col] = from_f32<T>(gate(g, u)); });
    } else if (UP) {
      ((T*)p.out)[(size_t)pair * p.n + col] = from_f32<T>(apply_act(acc[0][r], p.act));
    } else {
      float y = acc[0][r];
      if (!p.weight_on_input) y *= w;
      if (p.direct && p.residual) y += p.residual[(size_t)pair * p.n + col];
      ((float*)p.out)[(size_t)pair * p.n + col] = y;
    }
  }
}


// The same tile on the matrix unit, bfloat16 with an inner size in 8s: a wave takes 16 columns (and with GATED the
// 16 up rows that go with its 16 gate rows) for the tile's 16 pairs and makes out^T[column][pair] with MFMA
// 16x16x32, the matrix's rows as the A operand, the pairs' rows as the B operand. An expert's matrix is read once
// for every 16 of its pairs, which in a decode step is once, so what counts is how the matrix streams: a wave
// brings KC elements of each of its rows into a piece of LDS of its own with loads that cover a row's bytes side
// by side (512 bytes or more a row and instruction, marked as read once), all of a chunk's loads under way
// together, and takes the operands from there; the pairs' rows come from the caches. The waves of a block never
// wait for one another.
// PARTS: the waves of a block come in so many sets of four, each with its part of K; the sets' sums meet in LDS. Where a step
// is a few tokens an expert has one tile and a unit one block: with two sets there are twice as many loads under way, and half
// as many chunks one after the other (measured at `launch_products`).
// FOUND: up to 64 pairs, whose choices a wave holds: a block finds its expert and pairs in them, and no launch orders them
// first. Tiles are numbered without gaps, as the ordered ones are: blocks without one end at once, and where they stand between
// the others some units get two blocks and some none (4,096 wide, 8 pairs of 8 experts: 97 us a layer with a tile an expert
// whether it has pairs or not, 88.6 ordered).
template <int KIND, int PARTS, bool FOUND>
__global__ void __launch_bounds__(256 * PARTS) expert_product_mfma_kernel(ProductArgs p) {
  constexpr bool GATED = KIND == UP_GATED, UP = KIND != DOWN;
  constexpr int TM = 16;
  constexpr int ROWS = GATED ? 32 : 16;                   // rows of the matrix a wave holds
  constexpr int KC = 256;                                 // elements of K a chunk
  constexpr int LD = KC + 8;                              // a row in LDS: 16 bytes more, so that rows lie in different banks
  constexpr int LPR = KC / 8, RPI = 64 / LPR;             // lanes a row, rows an instruction
  constexpr int LOADS = ROWS / RPI;
  extern __shared__ __attribute__((aligned(16))) bf16_t staged[];     // [4 PARTS][ROWS * LD]
  __shared__ int pairs_of[FOUND ? TM : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const int part = PARTS > 1 ? __builtin_amdgcn_readfirstlane(wave >> 2) : 0, col0 = (blockIdx.x * 4 + (wave & 3)) * 16;
  int e = 0, pair;
  if constexpr (FOUND) {
    const int mine = lane < p.pairs ? p.chosen[lane] : -1;
    const bool counts = mine >= 0 && mine < p.experts;    // (beyond: an expert without tensors)
    const unsigned long long below = (1ull << lane) - 1;
    unsigned long long same = __ballot(counts);           // the lanes of the same expert, a bit of its number at a time
    for (int b = 0; 1 << b < p.experts; ++b) {
      const unsigned long long set = __ballot((mine >> b) & 1);
      same &= (mine >> b) & 1 ? set : ~set;
    }
    const int place = __popcll(same & below);             // among the pairs of its expert; every 16th begins a tile
    const bool begins = counts && place % TM == 0;
    const unsigned long long all = __ballot(begins);
    const unsigned long long its = __ballot(begins && __popcll(all & below) == (int)blockIdx.y);
    if (its == 0) return;
    const int from = __ffsll(its) - 1, begin = __shfl(place, from);
    e = __builtin_amdgcn_readfirstlane(__shfl(mine, from));
    const bool in = counts && mine == e && place >= begin && place < begin + TM;
    // (every wave writes the same numbers; a wave's LDS operations keep their order)
    if (in) pairs_of[place - begin] = lane;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    pair = r < __popcll(__ballot(in)) ? pairs_of[r] : -1;
  } else {
    int tile = blockIdx.y, begin = 0, end = 0;
    for (; e < p.experts; ++e) {
      begin = p.first[e];
      end = p.first[e + 1];
      const int tiles = (end - begin + TM - 1) / TM;
      if (tile < tiles) break;
      tile -= tiles;
    }
    if (e >= p.experts) return;
    begin += tile * TM;
    pair = begin + r < end ? p.order[begin + r] : -1;
  }
  if (PARTS == 1 && col0 >= p.n) return;
  float weight = 0.f;                                     // (asked for first where the pair is known at once)
  if (FOUND && pair >= 0) weight = p.weights[pair];
  const bf16_t* xrow = (const bf16_t*)p.a + (size_t)(pair < 0 ? 0 : (UP ? pair / p.top : pair)) * p.k;
  const bf16_t* W = (const bf16_t*)p.w + (size_t)e * (GATED ? 2 : 1) * p.n * p.k;
  bf16_t* mine = staged + wave * (ROWS * LD);
  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  // load i of a chunk: row RPI i + lane / LPR of the wave's rows (the up rows behind the gate rows), elements 8 (lane % LPR) on
  const int lrow = lane / LPR, lcol = 8 * (lane % LPR);
  const bf16_t* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = RPI * i + lrow;                       // 0 .. 15 gate (or plain) rows, 16 .. 31 up rows
    const int n = col0 + (row & 15);
    src[i] = n < p.n ? W + ((size_t)(row >> 4) * p.n + n) * p.k + lcol : nullptr;
  }
  const int chunks = (p.k + KC - 1) / KC, per = (chunks + PARTS - 1) / PARTS;
  const int k_begin = part * per * KC, k_end = min(p.k, k_begin + per * KC);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f}, acc_up = {0.f, 0.f, 0.f, 0.f};
  // a chunk's rows and the pair's elements that meet them are asked for while the chunk before is multiplied
  constexpr int STEPS = KC / 32;
  bf16x8 got[LOADS], x_next[STEPS];
  auto ask = [&](int k0) {
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int d = k0 + 32 * s + 8 * g;
      x_next[s] = (pair >= 0 && d < p.k) ? *(const bf16x8*)(xrow + d) : zero8;
    }
#pragma unroll
    for (int i = 0; i < LOADS; ++i) got[i] = (src[i] != nullptr && k0 + lcol < p.k) ? load_once(src[i] + k0) : zero8;
  };
  ask(k_begin);       // (a part beyond K asks for nothing; a branch around this made every load wait for the one before)
  for (int k0 = k_begin; k0 < k_end; k0 += KC) {
    bf16x8 x[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) x[s] = x_next[s];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) *(bf16x8*)(mine + (RPI * i + lrow) * LD + lcol) = got[i];
    if (k0 + KC < k_end) ask(k0 + KC);
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      if (k0 + 32 * s >= p.k) break;
      const int d0 = 32 * s + 8 * g;
      const bf16x8 a = *(const bf16x8*)(mine + r * LD + d0);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, x[s], acc, 0, 0, 0);
      if (GATED) {
        const bf16x8 u = *(const bf16x8*)(mine + (16 + r) * LD + d0);
        acc_up = __builtin_amdgcn_mfma_f32_16x16x32_bf16(u, x[s], acc_up, 0, 0, 0);
      }
    }
  }
  if (PARTS > 1) {
    // the later sets leave their sums in their own place in LDS, the first adds them in their order
    if (part > 0) {
      ((f32x4*)mine)[lane] = acc;
      if (GATED) ((f32x4*)mine)[64 + lane] = acc_up;
    }
    __syncthreads();
    if (part > 0) return;
#pragma unroll
    for (int q = 1; q < PARTS; ++q) {
      const f32x4* theirs = (const f32x4*)(staged + (wave + 4 * q) * (ROWS * LD));
      acc += theirs[lane];
      if (GATED) acc_up += theirs[64 + lane];
    }
  }
  if (pair < 0) return;
  if (!FOUND) weight = p.weights[pair];
  if constexpr (GATED)
    with_gate(p.act, p.limit, [&](auto gate) {
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = p.weight_on_input ? gate(acc[i] * weight, acc_up[i] * weight) : gate(acc[i], acc_up[i]);
    });
  else if constexpr (UP)
    with_act(p.act, [&](auto activation) {
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = activation(acc[i]);
    });
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int col = col0 + 4 * g + i;        // the lane holds columns 4 g .. 4 g + 3 of pair r
    if (col >= p.n) continue;
    if (UP) {
      ((bf16_t*)p.out)[(size_t)pair * p.n + col] = (bf16_t)acc[i];
    } else {
      float y = acc[i];
      if (!p.weight_on_input) y *= weight;
      if (p.direct && p.residual) y += p.residual[(size_t)pair * p.n + col];
      ((float*)p.out)[(size_t)pair * p.n + col] = y;
    }
  }
}

template <int KIND, int PARTS, bool FOUND>
int launch_products(const ProductArgs& p, dim3 grid, hipStream_t stream) {
  constexpr int bytes = 4 * PARTS * (KIND == UP_GATED ? 32 : 16) * (256 + 8) * 2;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void*)expert_product_mfma_kernel<KIND, PARTS, FOUND>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    TNX_REQUIRE(e == hipSuccess, "expert products: cannot reserve %d bytes of LDS: %s", bytes, hipGetErrorString(e));
    configured = true;
  }
  expert_product_mfma_kernel<KIND, PARTS, FOUND><<<grid, 256 * PARTS, bytes, stream>>>(p);
  return 0;
}

// Two sets of waves where K has two chunks for each and the blocks with a tile are at most one a unit: an expert has one tile
// where its pairs are few, ten on average at most; more, and some have two. Measured at two choices among 8 experts, us a layer
// with one set and with two: 2,048 wide, 1 token 45.6 / 31.7, 8 tokens 56.1 / 45.8 (256 blocks), 32 tokens 56.4 / 46.6, 33 tokens,
// 66 pairs, ordered first, 56.7 / 50.5, 48 tokens (96 pairs, 12 an expert) 67.5 / 73.9; 4,096 wide, 1 token (128 blocks) 73.9 / 59.5,
// 2 tokens (256) 80.5 / 70.2, 8 tokens (512) 151 / 166.
template <int KIND>
int launch_products(const ProductArgs& p, dim3 grid, hipStream_t stream) {
  const long long tiles = min(p.experts, p.pairs) + (p.pairs > 10 * p.experts ? p.pairs / 16 : 0);
  const bool two = p.k >= 1024 && grid.x * tiles <= tnx_compute_units();
  if (p.chosen) return two ? launch_products<KIND, 2, true>(p, grid, stream) : launch_products<KIND, 1, true>(p, grid, stream);
  return two ? launch_products<KIND, 2, false>(p, grid, stream) : launch_products<KIND, 1, false>(p, grid, stream);
}

// ---------------------------------------------------------------- many pairs an expert
// The same products where an expert has many pairs (prompts): tiles of 64 or 128 pairs by 128 or 256 of the matrix's rows on
// MFMA 32x32x16 (`tiles.h`), one launch over all experts. UP_GATED: a wave takes 32 gate rows and the 32 up rows that go with
// them, so that act(g) * u is made of its own sums; the tile makes half as many columns of `inner`. The pairs' rows are
// gathered by the loads themselves: a lane's address in `h` is that of its pair's token. `inner` and the result lie in sorted
// order. Of long prompts what bounds it is how well a unit's waves keep its matrix cores at work between their meetings (two waves
// a core and a wave's 64 x 64 of the tile: 60 % of the time), of short ones the bytes that a tile's block has to pull, 60 a nanosecond
// and unit while the matrices are in no cache (128 x 256 of K 2,048: 26 us, though it be on one unit in four). An expert's last
// tile may be nearly empty.
// Blocks of an XCD take the tiles of one column block after the other, so that an expert's rows of the matrix are brought
// from memory once and read again from that XCD's cache.
// Measured for 8 experts of which a token chooses two, a layer on weights that no cache holds, us, every tile whole / the last round in
// parts: 2,048 wide, inner 2,048: 64 tokens 75.2 / 59.9, 200 77.8 / 61.7, 396 83.0 / 75.0, 640 85.3 / 78.5, 1,024 113.8 / 106.5, 2,048 187 / 163;
// 4,096 wide, inner 4,096: 500 251 / 244, 1,000 344 / 318, 2,048 534 / 520 (790 TFLOP/s); 64 experts of 6, 2,048 wide, inner 1,408: 500
// 275 / 254, 2,048 438 / 410. Tiles of half or a quarter of the columns throughout are as much slower where whole ones go round the
// units more than once (2,048 wide, 2,048 tokens, halves: 197; 4,096 wide 575 to 630).
struct GroupedArgs {
  const bf16_t* a;          // UP: h [T, K]; DOWN: inner [sorted pairs, K]
  const bf16_t* w;          // [E, N(, 2), K]
  const int* first;         // [E + 1]
  const int* order;         // [pairs]
  const int2* tiles;        // [slots], then how many there are
  const float* weights;     // [pairs]; null: not on the input
  void* out;                // UP: inner, bfloat16; DOWN: float32
  int top, n, k, act, slots, units;
  float limit;
  int rows;                 // where there are no experts (`first`, `order` and `tiles` null): the rows of `a`, in their own order
};

// One tile: the pairs of `tile` by the columns of the result from n0 on.
template <int KIND, int MI, int NI, int ST, int WM, int WN>
__device__ __forceinline__ void expert_tile(const GroupedArgs& p, char* smem, const int2 tile, const int n0) {
  constexpr bool GATED = KIND == UP_GATED, UP = KIND != DOWN;
  static_assert(!GATED || NI == 2, "gate rows and the up rows beside them");
  typedef Tile<MI, NI, ST, WM, WN> Products;
  const int e = tile.x, begin = tile.y, count = min(Products::TM, (p.first ? p.first[e + 1] : p.rows) - begin);
  Products t;
#pragma unroll
  for (int j = 0; j < Products::LA; ++j) {
    const int row = Products::x_row(j), sorted = begin + min(row, count - 1);
    t.xoff[j] = 2u * ((unsigned)(UP && p.order ? p.order[sorted] / p.top : sorted) * (unsigned)p.k + Products::k_of(row));
  }
  const bf16_t* w = p.w + (size_t)e * (GATED ? 2 : 1) * p.n * p.k;
#pragma unroll
  for (int j = 0; j < Products::LB; ++j) {
    const int row = Products::w_row(j);
    // GATED: the tile's rows are, wave by wave, 32 gate rows and the 32 up rows beside them
    const int col = GATED ? n0 + 32 * (row >> 6) + (row & 31) : n0 + row;
    const unsigned from = (GATED && (row & 32) ? p.n : 0) + min(col, p.n - 1);
    t.woff[j] = 2u * (from * (unsigned)p.k + Products::k_of(row));
  }
  const int r0 = Products::row0(), c0 = n0 + (GATED ? Products::col0() / 2 : Products::col0());
  float weight[GATED ? MI : 1];      // (looked up before the products: at their end it would be two more times to reach memory)
  if constexpr (GATED) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
      weight[i] = p.weights ? p.weights[p.order[begin + min(r0 + 32 * i + (int)(threadIdx.x & 31), count - 1)]] : 1.f;
  }
  t.run(smem, p.a, w, p.k / 64);
  if constexpr (GATED) {
    with_gate(p.act, p.limit, [&](auto gate) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) t.acc[i][0][e] = gate(t.acc[i][0][e] * weight[i], t.acc[i][1][e] * weight[i]);
    });
    t.template hand_out<bf16_t, 32>(
        smem, [&](int i, int, int e, int, int) { return t.acc[i][0][e]; },
        [&](int r, int c, f32x4 chunk, int) {
          if (r0 + r < count && c0 + c < p.n) *(f32x4*)((bf16_t*)p.out + (size_t)(begin + r0 + r) * p.n + c0 + c) = chunk;
        });
  } else if constexpr (UP) {
    with_act(p.act, [&](auto activation) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) t.acc[i][j][e] = activation(t.acc[i][j][e]);
    });
    t.template hand_out<bf16_t, 32 * NI>(
        smem, [&](int i, int j, int e, int, int) { return t.acc[i][j][e]; },
        [&](int r, int c, f32x4 chunk, int) {
          if (r0 + r < count && c0 + c < p.n) *(f32x4*)((bf16_t*)p.out + (size_t)(begin + r0 + r) * p.n + c0 + c) = chunk;
        });
  } else {
    t.template hand_out<float, 32 * NI>(
        smem, [&](int i, int j, int e, int, int) { return t.acc[i][j][e]; },
        [&](int r, int c, f32x4 chunk, int) {
          if (r0 + r < count && c0 + c < p.n) *(f32x4*)((float*)p.out + (size_t)(begin + r0 + r) * p.n + c0 + c) = chunk;
        });
  }
}

// Tiles of 64 pairs: four waves over 128 rows of the matrix.
template <int KIND, int ST>
__global__ void __launch_bounds__(256) expert_tiles_kernel(GroupedArgs p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int at = by_xcd(blockIdx.x, gridDim.x);
  const int2 tile = p.tiles[at % p.slots];
  if (tile.x < 0) return;
  expert_tile<KIND, 1, 2, ST, 2, 2>(p, smem, tile, at / p.slots * (KIND == UP_GATED ? 64 : 128));
}

// Tiles of 128 pairs: eight waves over 256 rows of the matrix, as often as these go round the units, of which each holds one
// (144 KB). What is left over, less than one a unit, would be a whole round more for a part of the units: it goes out as halves
// or quarters of a tile's columns where these still find a unit each. How many tiles the pairs make only the device knows, so
// every block finds its place from their count.
template <int KIND>
__global__ void __launch_bounds__(512) expert_wide_tiles_kernel(GroupedArgs p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int COLUMNS = KIND == UP_GATED ? 128 : 256;
  auto tile = [&](int i) { return p.tiles ? p.tiles[i] : make_int2(0, 128 * i); };
  const int used = p.tiles ? p.tiles[p.slots].x : p.slots, total = used * ((p.n + COLUMNS - 1) / COLUMNS);
  int whole = total / p.units * p.units;
  const int left = total - whole;
  const int pieces = 4 * left <= p.units && KIND != UP_GATED ? 4 : 2 * left <= p.units ? 2 : 1;
  if (pieces == 1) whole = total;
  int block = blockIdx.x;
  if (block < whole) {
    const int at = by_xcd(block, whole);
    expert_tile<KIND, 2, 2, 3, 2, 4>(p, smem, tile(at % used), at / used * COLUMNS);
    return;
  }
  block -= whole;
  if (pieces == 1 || block >= left * pieces) return;
  const int piece = by_xcd(block, left * pieces), at = whole + piece / pieces;
  const int n0 = at / used * COLUMNS + piece % pieces * (COLUMNS / pieces);
  if (n0 >= p.n) return;
  if constexpr (KIND != UP_GATED) {
    if (pieces == 4) {
      expert_tile<KIND, 1, 1, 4, 4, 2>(p, smem, tile(at % used), n0);
      return;
    }
  }
  expert_tile<KIND, 1, 2, 4, 4, 2>(p, smem, tile(at % used), n0);
}

template <int KIND>
int launch_wide_tiles(const GroupedArgs& p, hipStream_t stream) {
  constexpr int bytes = Tile<2, 2, 3, 2, 4>::BYTES, columns = KIND == UP_GATED ? 128 : 256;
  static_assert(bytes >= Tile<1, 2, 4, 4, 2>::BYTES && bytes >= Tile<1, 1, 4, 4, 2>::BYTES, "room for the parts of a tile");
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void*)expert_wide_tiles_kernel<KIND>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    TNX_REQUIRE(e == hipSuccess, "expert tiles: cannot reserve %d bytes of LDS: %s", bytes, hipGetErrorString(e));
    configured = true;
  }
  // (whole rounds, and parts that fill one more at most)
  const long long total = (long long)((p.n + columns - 1) / columns) * p.slots, rounds = (total + p.units - 1) / p.units;
  expert_wide_tiles_kernel<KIND><<<(unsigned)(rounds * p.units), 512, bytes, stream>>>(p);
  TNX_CHECK_LAUNCH("expert tiles");
  return 0;
}

template <int KIND, int ST>
int launch_narrow_tiles(const GroupedArgs& p, hipStream_t stream) {
  constexpr int bytes = Tile<1, 2, ST, 2, 2>::BYTES, columns = KIND == UP_GATED ? 64 : 128;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void*)expert_tiles_kernel<KIND, ST>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    TNX_REQUIRE(e == hipSuccess, "expert tiles: cannot reserve %d bytes of LDS: %s", bytes, hipGetErrorString(e));
    configured = true;
  }
  expert_tiles_kernel<KIND, ST><<<(p.n + columns - 1) / columns * p.slots, 256, bytes, stream>>>(p);
  TNX_CHECK_LAUNCH("expert tiles");
  return 0;
}

// Tiles of 64 have two stages, so that a unit holds three blocks, four where it has no more than one anyway (the slots count an
// empty tile an expert too many, about half used).
template <int KIND>
int launch_tiles(const GroupedArgs& p, int tile_rows, hipStream_t stream) {
  if (tile_rows == 128) return launch_wide_tiles<KIND>(p, stream);
  const int columns = KIND == UP_GATED ? 64 : 128;
  const bool deep = (long long)((p.n + columns - 1) / columns) * p.slots <= p.units;
  return deep ? launch_narrow_tiles<KIND, 4>(p, stream) : launch_narrow_tiles<KIND, 2>(p, stream);
}

// (`place`: the row of y that holds pair t * top + c, where the rows lie in another order; `scale`: a factor a pair.
// With `same` a choice of `experts` or more is an expert without tensors: its row is the token's row of `same`, times the
// pair's weight.)
template <typename T, int V>
__global__ void combine_kernel(const float* __restrict__ y, const float* __restrict__ residual, float* __restrict__ out,
                               int top, int pieces, size_t total, const int* __restrict__ place,
                               const float* __restrict__ scale, const T* __restrict__ same,
                               const int* __restrict__ chosen, const float* __restrict__ weights, int experts) {
  typedef float fv __attribute__((ext_vector_type(V)));
  typedef T tv __attribute__((ext_vector_type(V)));
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < total; i += stride) {
    const size_t t = i / pieces, piece = i - t * pieces;
    fv s = 0.f;
    if (residual) s = ((const fv*)residual)[i];
    for (int c = 0; c < top; ++c) {
      const size_t pair = t * top + c;
      if (same && chosen[pair] >= experts) {
        const tv x = ((const tv*)same)[i];
#pragma unroll
        for (int e = 0; e < V; ++e) s[e] += weights[pair] * to_f32(x[e]);
        continue;
      }
      const fv v = ((const fv*)y)[(place ? (size_t)place[pair] : pair) * pieces + piece];
      const float w = scale ? scale[pair] : 1.f;
#pragma unroll
      for (int e = 0; e < V; ++e) s[e] += scale ? w * v[e] : v[e];
    }
    ((fv*)out)[i] = s;
  }
}

// act(g) * u from rows [g | u] of float32, V neighbours a thread (V = 4: halves of a multiple of four elements)
// (`row_weights`: a factor a row on both g and u, the weight on an expert's input)
// Memory bounds it: 2,048 rows of 2 x 8,192 are 168 MB and took 41 us one by one, 27 four by four.
template <typename T, int V>
__global__ void gated_activation_kernel(const float* __restrict__ gu, T* __restrict__ out, int pieces, int act, size_t total,
                                        const float* __restrict__ row_weights, float limit) {
  typedef float fv __attribute__((ext_vector_type(V)));
  typedef T tv __attribute__((ext_vector_type(V)));
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < total; i += stride) {
    const size_t t = i / pieces, at = i + t * pieces;       // piece i - t pieces of the row's first half
    const float w = row_weights ? row_weights[t] : 1.f;
    const fv g = ((const fv*)gu)[at], u = ((const fv*)gu)[at + pieces];
    tv o;
    with_gate(act, limit, [&](auto gate) {
#pragma unroll
      for (int e = 0; e < V; ++e) o[e] = from_f32<T>(gate(w * g[e], w * u[e]));
    });
    ((tv*)out)[i] = o;
  }
}

// act(x) from rows of float32 (`ld` apart), times sigmoid(row_gate) of the row; V neighbours a thread (V = 4: rows and
// places of a multiple of four elements)
template <typename T, int V>
__global__ void row_activation_kernel(const float* __restrict__ x, long long ld, T* __restrict__ out, int pieces, int act,
                                      size_t total, const float* __restrict__ row_gate, long long gate_ld) {
  typedef float fv __attribute__((ext_vector_type(V)));
  typedef T tv __attribute__((ext_vector_type(V)));
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < total; i += stride) {
    const size_t t = i / pieces, c = i - t * pieces;
    const fv v = *(const fv*)(x + t * ld + V * c);
    const float w = row_gate ? 1.f / (1.f + expf(-row_gate[t * gate_ld])) : 1.f;
    tv o;
    with_act(act, [&](auto activation) {
#pragma unroll
      for (int e = 0; e < V; ++e) o[e] = from_f32<T>(activation(v[e]) * w);
    });
    ((tv*)out)[i] = o;
  }
}

int blocks_for(size_t total) {
  size_t b = (total + 255) / 256;
  return (int)(b > 16384 ? 16384 : (b ? b : 1));
}

// The sum over a token's choices, four neighbours a thread where rows and places allow it.
template <typename T>
void launch_combine(const float* y, const float* residual, float* out, int tokens, int top, int width, const int* place,
                    const float* scale, const T* same, const int* chosen, const float* weights, int experts, hipStream_t stream) {
  const size_t total = (size_t)tokens * width;
  if (width % 4 == 0 && ((uintptr_t)y | (uintptr_t)residual | (uintptr_t)out | (uintptr_t)same) % 16 == 0)
    combine_kernel<T, 4><<<blocks_for(total / 4), 256, 0, stream>>>(y, residual, out, top, width / 4, total / 4, place, scale, same,
                                                                     chosen, weights, experts);
  else
    combine_kernel<T, 1><<<blocks_for(total), 256, 0, stream>>>(y, residual, out, top, width, total, place, scale, same, chosen,
                                                                 weights, experts);
}

}  // namespace

extern "C" int tnx_route(const float* z, int ld, int tokens, int experts, int top, int softmax, int renormalize, int* chosen,
                         float* weights, const float* correction, float scale, int groups, int keep, hipStream_t stream) {
  TNX_REQUIRE(tokens >= 0 && experts > 0 && top > 0 && top <= experts, "route: %d of %d experts", top, experts);
  TNX_REQUIRE(ld >= experts, "route: rows of %d logits, %d experts", ld, experts);
  TNX_REQUIRE(experts <= 4096, "route: up to 4096 experts, got %d", experts);
  TNX_REQUIRE(groups >= 1 && groups <= MAX_GROUPS && experts % groups == 0 && keep >= 1 && keep <= groups &&
                  top <= keep * (experts / groups),
              "route: %d of %d experts in %d groups (up to %d) of which %d are kept", top, experts, groups, MAX_GROUPS, keep);
  if (tokens == 0) return 0;
  route_kernel<<<(tokens + 3) / 4, 256, 0, stream>>>(
      z, ld, RouteArgs{tokens, experts, top, softmax, renormalize, chosen, weights, correction, scale, groups, keep});
  TNX_CHECK_LAUNCH("route");
  return 0;
}

// The same from the rows `h` [tokens, width] and the router's matrix `w` [experts, width], bfloat16, and its bias or none.
extern "C" int tnx_route_product(const void* h, const void* w, const float* bias, int width, int tokens, int experts, int top,
                                 int softmax, int renormalize, int* chosen, float* weights, const float* correction, float scale,
                                 int groups, int keep, hipStream_t stream) {
  TNX_REQUIRE(tokens >= 0 && experts > 0 && top > 0 && top <= experts, "route_product: %d of %d experts", top, experts);
  TNX_REQUIRE(experts <= ROUTE_PRODUCT_MOST, "route_product: up to %d experts, got %d", ROUTE_PRODUCT_MOST, experts);
  TNX_REQUIRE(width > 0 && width % 8 == 0 && ((uintptr_t)h | (uintptr_t)w) % 16 == 0, "route_product: rows of %d, in 8s and 16-byte aligned", width);
  TNX_REQUIRE(groups >= 1 && experts % groups == 0 && keep >= 1 && keep <= groups && top <= keep * (experts / groups),
              "route_product: %d of %d experts in %d groups of which %d are kept", top, experts, groups, keep);
  if (tokens == 0) return 0;
  route_product_kernel<<<tokens, 256, 0, stream>>>(
      (const bf16_t*)h, (const bf16_t*)w, bias, width,
      RouteArgs{tokens, experts, top, softmax, renormalize, chosen, weights, correction, scale, groups, keep});
  TNX_CHECK_LAUNCH("route_product");
  return 0;
}

// (`out` null: the pairs' weighted rows stay in `pair_rows`, for a product that adds them.)
extern "C" int tnx_expert_mixture(const void* h, const int* chosen, const float* weights, const void* w_gate_up,
                                  const void* w_down, int* first, int* order, void* inner, float* pair_rows,
                                  const float* residual, float* out, int dtype, int tokens, int experts, int top,
                                  int width, int f, int act, int weight_on_input, int plain, float limit,
                                  int identity, int ungated, hipStream_t stream) {
  TNX_REQUIRE(!ungated || !weight_on_input, "expert_mixture: experts without a gate take their weight on the output");
  TNX_REQUIRE(tokens >= 0 && experts > 0 && top > 0 && width > 0 && f > 0, "expert_mixture: bad sizes");
  TNX_REQUIRE(experts <= 4096, "expert_mixture: up to 4096 experts, got %d", experts);
  TNX_REQUIRE(dtype == TNX_F32 || dtype == TNX_BF16, "expert_mixture: dtype %d", dtype);
  const bool direct = top == 1 && !identity;
  TNX_REQUIRE(out != nullptr || (!direct && !identity), "expert_mixture: only pairs' rows of experts with tensors are left to their reader");
  TNX_REQUIRE(direct || pair_rows != nullptr, "expert_mixture: several choices a token need room for their rows");
  TNX_REQUIRE(!identity || !weight_on_input, "expert_mixture: experts without tensors take their weight on the output");
  if (tokens == 0) return 0;
  const int pairs = tokens * top;
  const bool mfma = dtype == TNX_BF16 && width % 8 == 0 && f % 8 == 0 && !plain;
  // Up to 64 pairs the products' blocks find their pairs themselves (a wave holds all choices), which saves the launch that
  // orders them (3 to 4 us).
  const bool found = mfma && pairs <= 64;
  if (!found) {
    order_kernel<<<1, 1024, 2 * experts * sizeof(int), stream>>>(chosen, pairs, experts, first, order, nullptr, nullptr, top,
                                                                 nullptr, nullptr, nullptr, 0, 0);
    TNX_CHECK_LAUNCH("expert order");
  }
  // the most tiles of 16 pairs: every expert that has pairs may end in a part of one
  const int tiles = pairs / 16 + min(experts, pairs);
  const int* look = found ? chosen : nullptr;
  ProductArgs up{h, w_gate_up, first, order, weights, nullptr, inner, experts, top, f, width, act, weight_on_input, pairs,
                 limit, 0, look};
  ProductArgs down{inner, w_down, first, order, weights, residual, direct ? out : pair_rows, experts, top, width, f,
                   act, weight_on_input, pairs, limit, direct ? 1 : 0, look};
  const dim3 grid_up((f + 63) / 64, tiles), grid_down((width + 63) / 64, tiles);
  if (dtype == TNX_F32) {
    if (ungated)
      expert_product_kernel<float, UP_PLAIN><<<grid_up, 256, 0, stream>>>(up);
    else
      expert_product_kernel<float, UP_GATED><<<grid_up, 256, 0, stream>>>(up);
    expert_product_kernel<float, DOWN><<<grid_down, 256, 0, stream>>>(down);
  } else if (mfma) {
    if (int rc = ungated ? launch_products<UP_PLAIN>(up, grid_up, stream) : launch_products<UP_GATED>(up, grid_up, stream)) return rc;
    if (int rc = launch_products<DOWN>(down, grid_down, stream)) return rc;
  } else {
    if (ungated)
      expert_product_kernel<bf16_t, UP_PLAIN><<<grid_up, 256, 0, stream>>>(up);
    else
      expert_product_kernel<bf16_t, UP_GATED><<<grid_up, 256, 0, stream>>>(up);
    expert_product_kernel<bf16_t, DOWN><<<grid_down, 256, 0, stream>>>(down);
  }
  TNX_CHECK_LAUNCH("expert products");
  if (!direct && out) {
    if (dtype == TNX_F32)
      launch_combine<float>(pair_rows, residual, out, tokens, top, width, nullptr, nullptr, identity ? (const float*)h : nullptr,
                            chosen, weights, experts, stream);
    else
      launch_combine<bf16_t>(pair_rows, residual, out, tokens, top, width, nullptr, nullptr,
                             identity ? (const bf16_t*)h : nullptr, chosen, weights, experts, stream);
    TNX_CHECK_LAUNCH("expert combine");
  }
  return 0;
}

// The whole mixture for many pairs an expert, in bfloat16: order, the two products by tiles of `tile_rows` (64 or 128) pairs,
// the sum. `ints`: room for experts + 1 + 2 pairs integers, then 2 (pairs / tile_rows + experts + 1) more from a multiple of 2 on;
// `inner` [pairs, f], `y` [pairs, width]. width and f are multiples of 64.
extern "C" int tnx_expert_grouped(const void* h, const int* chosen, const float* weights, const void* w_gate_up,
                                  const void* w_down, int* ints, void* inner, float* y, const float* residual, float* out,
                                  int tokens, int experts, int top, int width, int f, int act, int weight_on_input, float limit,
                                  int identity, int ungated, int tile_rows, hipStream_t stream) {
  TNX_REQUIRE(!ungated || !weight_on_input, "expert_grouped: experts without a gate take their weight on the output");
  TNX_REQUIRE(!identity || !weight_on_input, "expert_grouped: experts without tensors take their weight on the output");
  TNX_REQUIRE(tokens >= 0 && experts > 0 && experts <= 4096 && top > 0, "expert_grouped: bad sizes");
  TNX_REQUIRE(width > 0 && f > 0 && width % 64 == 0 && f % 64 == 0, "expert_grouped: sizes in 64s, got %d and %d", width, f);
  TNX_REQUIRE(tile_rows == 64 || tile_rows == 128, "expert_grouped: tiles of 64 or 128 pairs");
  TNX_REQUIRE((long long)tokens * top < (1ll << 30), "expert_grouped: too many pairs");
  TNX_REQUIRE((long long)tokens * width < (1ll << 31) && (long long)tokens * top * f < (1ll << 31) &&
                  (long long)width * f < (1ll << 30), "expert_grouped: operands of 4 GB or more");
  TNX_REQUIRE(((uintptr_t)h | (uintptr_t)w_gate_up | (uintptr_t)w_down | (uintptr_t)inner | (uintptr_t)y) % 16 == 0 &&
                  (uintptr_t)ints % 8 == 0, "expert_grouped: operands must be 16-byte aligned");
  if (tokens == 0) return 0;
  const int pairs = tokens * top, slots = pairs / tile_rows + experts;      // every expert may end in a part of a tile
  TNX_REQUIRE((long long)slots * ((width > f ? width : f) / 64 + 1) < (1ll << 31), "expert_grouped: too many tiles");
  int *first = ints, *order = first + experts + 1, *place = order + pairs;
  int2* tiles = (int2*)(ints + (experts + 1 + 2 * (size_t)pairs + 1) / 2 * 2);
  order_kernel<<<1, 1024, 3 * experts * sizeof(int), stream>>>(chosen, pairs, experts, first, order, place, nullptr, top, nullptr,
                                                               nullptr, tiles, tile_rows, slots);
  TNX_CHECK_LAUNCH("expert order");
  const GroupedArgs up{(const bf16_t*)h, (const bf16_t*)w_gate_up, first, order, tiles, weight_on_input ? weights : nullptr, inner,
                       top, f, width, act, slots, tnx_compute_units(), limit, 0};
  const GroupedArgs down{(const bf16_t*)inner, (const bf16_t*)w_down, first, order, tiles, nullptr, y, top, width, f, act, slots,
                         tnx_compute_units(), limit, 0};
  if (int rc = ungated ? launch_tiles<UP_PLAIN>(up, tile_rows, stream) : launch_tiles<UP_GATED>(up, tile_rows, stream)) return rc;
  if (int rc = launch_tiles<DOWN>(down, tile_rows, stream)) return rc;
  launch_combine<bf16_t>(y, residual, out, tokens, top, width, place, weight_on_input ? nullptr : weights,
                         identity ? (const bf16_t*)h : nullptr, chosen, weights, experts, stream);
  TNX_CHECK_LAUNCH("expert combine");
  return 0;
}

extern "C" int tnx_gated_activation(const float* gate_up, void* out, int dtype, int tokens, int f, int act,
                                    const float* row_weights, float limit, hipStream_t stream) {
  TNX_REQUIRE(tokens >= 0 && f > 0, "gated_activation: bad sizes");
  TNX_REQUIRE(dtype == TNX_F32 || dtype == TNX_BF16, "gated_activation: dtype %d", dtype);
  if (tokens == 0) return 0;
  const size_t total = (size_t)tokens * f;
  // (fewer elements than threads the units hold half of: one a thread. 33 rows of 4,096 2.64 us, four a thread 2.96; 33 of 8,192
  // 3.00 and 3.00, 100 of 4,096 3.36 and 3.08.)
  const bool fours = f % 4 == 0 && (uintptr_t)gate_up % 16 == 0 && (uintptr_t)out % (dtype == TNX_F32 ? 16 : 8) == 0 &&
                     total > (size_t)1024 * tnx_compute_units();
#define GATED_LAUNCH(T, V)                                                                                              \
  gated_activation_kernel<T, V><<<blocks_for(total / V), 256, 0, stream>>>(gate_up, (T*)out, f / V, act, total / V,      \
                                                                           row_weights, limit)
  if (dtype == TNX_F32) {
    if (fours) GATED_LAUNCH(float, 4);
    else GATED_LAUNCH(float, 1);
  } else {
    if (fours) GATED_LAUNCH(bf16_t, 4);
    else GATED_LAUNCH(bf16_t, 1);
  }
#undef GATED_LAUNCH
  TNX_CHECK_LAUNCH("gated_activation");
  return 0;
}

// act(g) * u from the rows x [tokens, width] and w [2 f, width] (gate rows, then up rows), bfloat16, by the experts' tiles: the sums
// stay in registers until both halves are there.
extern "C" int tnx_gated_activation_tiles(const void* x, const void* w, void* out, int act, float limit, int tokens, int f, int width,
                                          hipStream_t stream) {
  TNX_REQUIRE(tokens >= 0 && f > 0 && width > 0 && width % 64 == 0 && f % 64 == 0, "gated_activation_tiles: sizes in 64s, got %d and %d", width, f);
  TNX_REQUIRE((long long)tokens * width < (1ll << 31) && (long long)width * f < (1ll << 30) && (long long)tokens * f < (1ll << 31),
              "gated_activation_tiles: operands of 4 GB or more");
  TNX_REQUIRE(((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) % 16 == 0, "gated_activation_tiles: operands must be 16-byte aligned");
  if (tokens == 0) return 0;
  const int slots = (tokens + 127) / 128;
  TNX_REQUIRE((long long)slots * (f / 64 + 1) < (1ll << 31) - 1024, "gated_activation_tiles: too many tiles");
  return launch_wide_tiles<UP_GATED>(GroupedArgs{(const bf16_t*)x, (const bf16_t*)w, nullptr, nullptr, nullptr, nullptr, out, 1, f, width, act,
                                                 slots, tnx_compute_units(), limit, tokens}, stream);
}

// act(x) of float32 rows (`ld` apart), times sigmoid(row_gate) of its row (numbers `gate_ld` apart) or not
extern "C" int tnx_row_activation(const float* x, long long ld, void* out, int dtype, int tokens, int f, int act,
                                  const float* row_gate, long long gate_ld, hipStream_t stream) {
  TNX_REQUIRE(tokens >= 0 && f > 0 && ld >= f && gate_ld >= 0, "row_activation: bad sizes");
  TNX_REQUIRE(dtype == TNX_F32 || dtype == TNX_BF16, "row_activation: dtype %d", dtype);
  if (tokens == 0) return 0;
  const size_t total = (size_t)tokens * f;
  const bool fours = f % 4 == 0 && ld % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)out % (dtype == TNX_F32 ? 16 : 8) == 0;
#define ROWS_LAUNCH(T, V) \
  row_activation_kernel<T, V><<<blocks_for(total / V), 256, 0, stream>>>(x, ld, (T*)out, f / V, act, total / V, row_gate, gate_ld)
  if (dtype == TNX_F32) {
    if (fours) ROWS_LAUNCH(float, 4);
    else ROWS_LAUNCH(float, 1);
  } else {
    if (fours) ROWS_LAUNCH(bf16_t, 4);
    else ROWS_LAUNCH(bf16_t, 1);
  }
#undef ROWS_LAUNCH
  TNX_CHECK_LAUNCH("row_activation");
  return 0;
}

// The pairs in the order of their experts, for a caller that runs the experts' products itself: `first[E + 1]`,
// `order[pairs]`, `place[pairs]` (where a pair went), `token[pairs]` (the token of each sorted row) and the weights in
// sorted order.
extern "C" int tnx_expert_order(const int* chosen, const float* weights, int tokens, int experts, int top, int* first,
                                int* order, int* place, int* token, float* sorted_weights, hipStream_t stream) {
  TNX_REQUIRE(tokens >= 0 && experts > 0 && experts <= 4096 && top > 0, "expert_order: bad sizes");
  if (tokens == 0) return 0;
  order_kernel<<<1, 1024, 2 * experts * sizeof(int), stream>>>(chosen, tokens * top, experts, first, order, place, token,
                                                               top, weights, sorted_weights, nullptr, 0, 0);
  TNX_CHECK_LAUNCH("expert order");
  return 0;
}

// out[t] = residual[t] + sum_c scale[t, c] y[place[t * top + c]]; with `same` (bfloat16 rows) a choice of `experts` or more
// adds scale[t, c] same[t]
extern "C" int tnx_expert_combine(const float* y, const int* place, const float* scale, const float* residual, float* out,
                                  int tokens, int top, int width, const void* same, const int* chosen, int experts,
                                  hipStream_t stream) {
  TNX_REQUIRE(tokens >= 0 && top > 0 && width > 0, "expert_combine: bad sizes");
  if (tokens == 0) return 0;
  TNX_REQUIRE(!same || (scale && chosen), "expert_combine: experts without tensors need the choices and their weights");
  launch_combine<bf16_t>(y, residual, out, tokens, top, width, place, scale, (const bf16_t*)same, chosen, scale, experts, stream);
  TNX_CHECK_LAUNCH("expert combine");
  return 0;
}
