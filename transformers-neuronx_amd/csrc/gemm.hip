// Matrix products `out[M, N] = act(x[M, K] w[N, K]^T + bias[N]) + residual[M, N]` with float32 accumulation.
//   gemm_f32        float32 operands, as three bfloat16 parts each on the matrix instructions (nothing of an operand is lost), on
//                   plain FMA for few rows and for sizes that are no multiples of 32 in K
//   gemm_bf16       bfloat16 operands on MFMA, many rows (prompts): 256x256x64 tiles, operands straight from
//                   global memory into two LDS stages, four waves of 128x128 (sizes in whole 64-steps of K);
//                   128x128 tiles staged through registers for every other size
//   gemm_bf16_skinny  bfloat16 operands on MFMA for M <= 64 (decoding): streams the weight once
// bias and residual are float32 and optional; the output is float32 or bfloat16.
#include "tiles.h"
#include <type_traits>

TNX_DEFINE_ERROR_API


__device__ __forceinline__ void epilogue_store(float v, int m, int n, int N, const float* bias, const float* residual,
                                               void* out, int out_dtype, int act) {
  if (bias) v += bias[n];
  v = apply_act(v, act);
  const size_t o = (size_t)m * N + n;
  if (residual) v += residual[o];
  store_any(out, out_dtype, o, v);
}

// Where the fused query/key/value projection puts its output: queries (scaled) into a dense matrix, the
// keys and values of token m into the cache page `token_page[m]` at place `token_off[m]`
// (keys [pages, kv_heads, page_size, head_size], values [pages, kv_heads, head_size, page_size]).
// `turn_a`, `turn_b` (both or neither): a position encoding that turns queries and keys pair by pair, as
// tables [turn_rows, head_size] of float32. Element d of a query or key head of the token at position p
// becomes a[p][d] x[d] + b[p][d] x[d ^ 1], bias added, before the query's scale: any map of each pair
// (2i, 2i + 1) of a head that depends on the position alone (a rotation: a = cos, b = -sin and +sin).
template <typename T>
struct QkvScatterOf {
  const int* token_page;
  const int* token_off;
  T* q_out;
  T* k_pages;
  T* v_pages;
  float scale;
  int nq, nk, head_size, num_kv, page_size, num_pages;
  int page_pad;          // elements between the end of one page and the start of the next
  const float* turn_a;
  const float* turn_b;
  const int* positions;
  int turn_rows;
};
typedef QkvScatterOf<bf16_t> QkvScatter;
struct NoScatter {};

// `v`: element n of token m's projections with its bias; `beside`: element n ^ 1 with its bias (read only
// where the scatter turns pairs)
// (`page`, `off`: what `token_page` and `token_off` say of token m)
template <typename T>
__device__ __forceinline__ void qkv_store(float v, float beside, int m, int n, const QkvScatterOf<T>& sc, int page, int off) {
  if (sc.turn_a && n < sc.nq + sc.nk) {
    const size_t at = (size_t)min(max(sc.positions[m], 0), sc.turn_rows - 1) * sc.head_size + n % sc.head_size;
    v = sc.turn_a[at] * v + sc.turn_b[at] * beside;
  }
  if (n < sc.nq) {
    sc.q_out[(size_t)m * sc.nq + n] = from_f32<T>(v * sc.scale);
    return;
  }
  if (page < 0 || page >= sc.num_pages) return;
  int j = n - sc.nq;
  const bool is_key = j < sc.nk;
  if (!is_key) j -= sc.nk;
  const int h = j / sc.head_size, d = j - h * sc.head_size;
  const size_t head_elems = (size_t)sc.page_size * sc.head_size;
  const size_t head = (size_t)page * ((size_t)sc.num_kv * head_elems + sc.page_pad) + (size_t)h * head_elems;
  if (is_key)
    sc.k_pages[head + (size_t)off * sc.head_size + d] = from_f32<T>(v);
  else
    sc.v_pages[head + (size_t)d * sc.page_size + off] = from_f32<T>(v);
}

// Four neighbouring elements of a result (`fours`: they lie where one store can put them).
__device__ __forceinline__ void store_four(f32x4 v, void* out, int out_dtype, size_t o, bool fours) {
  if (!fours) {
#pragma unroll
    for (int e = 0; e < 4; ++e) store_any(out, out_dtype, o + e, v[e]);
  } else if (out_dtype == TNX_F32) {
    *(f32x4*)((float*)out + o) = v;
  } else {
    bf16x4 b;
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = (bf16_t)v[e];
    *(bf16x4*)((bf16_t*)out + o) = b;
  }
}

// Whether `qkv_store_four` may be asked: heads in fours, so that four columns are all queries', keys' or values', of one head,
// and everything where four elements are read or written at once (pages lie multiples of 8 elements apart).
__device__ __forceinline__ bool qkv_in_fours(const QkvScatter& sc) {
  return sc.head_size % 4 == 0 && (((uintptr_t)sc.q_out | (uintptr_t)sc.k_pages) & 7) == 0 &&
         (((uintptr_t)sc.turn_a | (uintptr_t)sc.turn_b) & 15) == 0;
}

// `qkv_store` of columns n .. n + 3 (n a multiple of 4), the same results.
__device__ __forceinline__ void qkv_store_four(f32x4 v, int m, int n, const QkvScatter& sc, int page, int off) {
  if (sc.turn_a && n < sc.nq + sc.nk) {
    const size_t at = (size_t)min(max(sc.positions[m], 0), sc.turn_rows - 1) * sc.head_size + n % sc.head_size;
    const f32x4 a = *(const f32x4*)(sc.turn_a + at), b = *(const f32x4*)(sc.turn_b + at);
    v = a * v + b * (f32x4){v[1], v[0], v[3], v[2]};
  }
  if (n < sc.nq) v *= sc.scale;
  bf16x4 four;
#pragma unroll
  for (int e = 0; e < 4; ++e) four[e] = (bf16_t)v[e];
  if (n < sc.nq) {
    *(bf16x4*)(sc.q_out + (size_t)m * sc.nq + n) = four;
    return;
  }
  if (page < 0 || page >= sc.num_pages) return;
  int j = n - sc.nq;
  const bool is_key = j < sc.nk;
  if (!is_key) j -= sc.nk;
  const int h = j / sc.head_size, d = j - h * sc.head_size;
  const size_t head_elems = (size_t)sc.page_size * sc.head_size;
  const size_t head = (size_t)page * ((size_t)sc.num_kv * head_elems + sc.page_pad) + (size_t)h * head_elems;
  if (is_key) {
    *(bf16x4*)(sc.k_pages + head + (size_t)off * sc.head_size + d) = four;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) sc.v_pages[head + (size_t)(d + e) * sc.page_size + off] = four[e];
  }
}

// ------------------------------------------------------------------------------------------ float32

#define F32_TILE 64
#define F32_BK 16

__global__ void __launch_bounds__(256)
gemm_f32_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
                const float* __restrict__ residual, void* __restrict__ out, int out_dtype, int act, int M, int N,
                int K) {
  __shared__ float xs[F32_BK][F32_TILE + 4];
  __shared__ float ws[F32_BK][F32_TILE + 4];
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  const int m0 = blockIdx.y * F32_TILE, n0 = blockIdx.x * F32_TILE;
  const int lrow = tid >> 2, lk = (tid & 3) * 4;  // this thread stages row lrow, k lk..lk+3 of both tiles
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  for (int k0 = 0; k0 < K; k0 += F32_BK) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = k0 + lk + e;
      const int m = m0 + lrow, n = n0 + lrow;
      xs[lk + e][lrow] = (m < M && k < K) ? x[(size_t)m * K + k] : 0.f;
      ws[lk + e][lrow] = (n < N && k < K) ? w[(size_t)n * K + k] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < F32_BK; ++k) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = xs[k][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = ws[k][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n < N) epilogue_store(acc[i][j], m, n, N, bias, residual, out, out_dtype, act);
    }
  }
}

// Few rows in float32 (decoding): the product is the weight read once. A wave makes 4 columns of the output
// for up to MR rows of `x`; its lanes share K four floats at a time, so a row of the weight is read in runs
// of 1 KB, and the 64 partial sums of every output meet in a butterfly at the end. K is a multiple of 4.
// SPLIT: the block's four waves make the same 4 columns and take steps of 256 of K in turn, their sums meet in LDS; where
// the columns are few, four times the blocks read the weight and a wave's chain of waits is a quarter as long. UNROLL steps
// are asked for together: what bounds a narrow matrix is how often a wave waits for memory, not the bytes. Measured at 3
// rows, a wave for every 4 columns against four: 1,024 columns of K 4,096 13.8 us against 7.7, 4,096 of 1,024 9.8 against 8.3;
// with bias and residual asked for first and the weight marked as read once 6.8 and 7.6.
// Scatter (`QkvScatterOf<float>`): queries, keys and values go where they belong from here, in place of a matrix that another
// launch reads again. 3 rows of 3,072 by 1,024: 7.3 us, where the product took 6.5 and the other launch 3.2.
template <int MR, bool SPLIT, int UNROLL, typename Scatter>
__global__ void __launch_bounds__(256)
gemm_f32_skinny_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
                       const float* __restrict__ residual, void* __restrict__ out, int out_dtype, int act, int M,
                       int N, int K, Scatter sc) {
  constexpr bool SCATTER = !std::is_same<Scatter, NoScatter>::value;
  __shared__ float sums[SPLIT ? 4 : 1][4 * MR];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = (SPLIT ? blockIdx.x : blockIdx.x * 4 + wave) * 4;
  if (n0 >= N) return;                 // (SPLIT: the whole block)
  const float* wrow[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) wrow[c] = w + (size_t)min(n0 + c, N - 1) * K;
  const float* xrow[MR];
#pragma unroll
  for (int m = 0; m < MR; ++m) xrow[m] = x + (size_t)min(m, M - 1) * K;
  // bias and residual of the element that this thread puts out, asked for before anything else
  const int put = SPLIT ? threadIdx.x : lane, put_c = n0 + put / MR, put_m = put % MR;
  const bool puts = put < 4 * MR && put_c < N && put_m < M;
  float add = 0.f, onto = 0.f;
  if (puts && bias) add = bias[put_c];
  if (puts && residual) onto = residual[(size_t)put_m * N + put_c];
  int page = -1, off = 0;
  if constexpr (SCATTER) {
    if (puts) page = sc.token_page[put_m], off = sc.token_off[put_m];
  }
  float acc[4][MR];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[c][m] = 0.f;
  const int k_last = K - 4;
  constexpr int STRIDE = SPLIT ? 1024 : 256;
  for (int k0 = SPLIT ? 256 * wave : 0; k0 < K; k0 += STRIDE * UNROLL) {
    f32x4 wv[UNROLL][4], xv[UNROLL][MR];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      // lanes beyond K read the last four floats again and add nothing
      const int k = min(k0 + u * STRIDE + 4 * lane, k_last);
#pragma unroll
      for (int c = 0; c < 4; ++c) wv[u][c] = __builtin_nontemporal_load((const f32x4*)(wrow[c] + k));
#pragma unroll
      for (int m = 0; m < MR; ++m) xv[u][m] = *(const f32x4*)(xrow[m] + k);
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      if (k0 + u * STRIDE + 4 * lane >= K) continue;
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int m = 0; m < MR; ++m) {
          float a = acc[c][m];
          a = fmaf(wv[u][c][0], xv[u][m][0], a);
          a = fmaf(wv[u][c][1], xv[u][m][1], a);
          a = fmaf(wv[u][c][2], xv[u][m][2], a);
          a = fmaf(wv[u][c][3], xv[u][m][3], a);
          acc[c][m] = a;
        }
    }
  }
  // every lane gets a sum; lane c * MR + m keeps that of column c, row m
  float mine = 0.f;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const float a = wave_sum(acc[c][m]);
      if (lane == c * MR + m) mine = a;
    }
  if (SPLIT) {
    if (lane < 4 * MR) sums[wave][lane] = mine;
    __syncthreads();
    if (puts) mine = (sums[0][put] + sums[1][put]) + (sums[2][put] + sums[3][put]);
  }
  if constexpr (SCATTER) {
    if (bias) mine += add;
    const float beside = __shfl_xor(mine, MR);          // column c ^ 1 of the same row
    if (puts) qkv_store(mine, beside, put_m, put_c, sc, page, off);
  } else if (puts) {
    float v = mine;
    if (bias) v += add;
    v = apply_act(v, act);
    if (residual) v += onto;
    store_any(out, out_dtype, (size_t)put_m * N + put_c, v);
  }
}

template <int MR, typename Scatter>
static void launch_f32_skinny(const float* x, const float* w, const float* bias, const float* residual, void* out,
                              int out_dtype, int act, int M, int N, int K, const Scatter& sc, hipStream_t stream) {
  // Steps asked for together: as many as the rows leave registers for.
  constexpr int MOST = MR <= 4 ? 4 : MR <= 8 ? 2 : 1;
#define SKINNY_F32(SPLIT, UNROLL, GRID)                                                                            \
  gemm_f32_skinny_kernel<MR, SPLIT, UNROLL, Scatter><<<dim3(GRID), 256, 0, stream>>>(x, w, bias, residual, out,     \
                                                                                     out_dtype, act, M, N, K, sc)
  // A wave for every 4 columns gives N / 16 blocks; below four blocks a compute unit the waves of a block share K instead.
  if ((N + 15) / 16 < 4 * tnx_compute_units()) {
    if (K > 1024 && MOST > 1)
      SKINNY_F32(true, MOST, (N + 3) / 4);
    else
      SKINNY_F32(true, 1, (N + 3) / 4);
  } else {
    SKINNY_F32(false, (MOST > 2 ? 2 : MOST), (N + 15) / 16);
  }
#undef SKINNY_F32
}

// By the number of rows, up to 16.
template <typename Scatter>
static void f32_skinny(const float* x, const float* w, const float* bias, const float* residual, void* out, int out_dtype,
                       int act, int M, int N, int K, const Scatter& sc, hipStream_t stream) {
  if (M <= 1)
    launch_f32_skinny<1>(x, w, bias, residual, out, out_dtype, act, M, N, K, sc, stream);
  else if (M <= 2)
    launch_f32_skinny<2>(x, w, bias, residual, out, out_dtype, act, M, N, K, sc, stream);
  else if (M <= 4)
    launch_f32_skinny<4>(x, w, bias, residual, out, out_dtype, act, M, N, K, sc, stream);
  else if (M <= 8)
    launch_f32_skinny<8>(x, w, bias, residual, out, out_dtype, act, M, N, K, sc, stream);
  else
    launch_f32_skinny<16>(x, w, bias, residual, out, out_dtype, act, M, N, K, sc, stream);
}

// Many rows in float32, on the bfloat16 matrix instructions: every operand is the sum of three bfloat16 parts, x = h + m + l
// with h = x rounded, m = (x - h) rounded and l the rest, which eight bits hold: nothing of x is lost. Of the nine products of
// parts six are made, each exact, with float32 sums (the scheme of Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial
// intelligence datatype for higher-precision computations", 2019); l l, l m and m l are left out: |m| is at most 2^-8 and |l| 2^-17
// of |x|, which makes them 2^-24 of |x w| between them, as much again as a rounding of the product. A result of one product is thus
// off by up to twice that rounding, where the float32 instructions made one; on average it is as near, and a sum of many is nearer
// (below). Operands under 2^-110 lose more, what of a lower part is under the smallest bfloat16 number: up to 2^-134 of themselves.
// The float32 instructions give 256 flops a cycle and unit, the bfloat16 ones 4,096, of which a sixth is 683.
// h h has sums of its own, the other five share theirs: six times fewer roundings at the size of the result, which is why the
// error against 64 bits is 0.34 to 0.7 of what the float32 instructions left (K 2,048: 2.7e-7 for 8.1e-7, 1,024: 1.9e-7 for 5.7e-7;
// with one set of sums for all six 7.0e-7).
// Tiles of 32 MI WM rows of `x` by 32 NI WN of `w`, 32 of K a step. A thread loads rows three steps ahead into registers, splits
// them beside the products of the two steps before their own and leaves the parts in LDS, two stages of them (a split wave by
// wave, from float32 in LDS, would be made again by every wave that shares the rows). Of a step of 128 x 128 the matrix cores
// need 0.64 us; it takes 0.89 with a block on every fourth unit and 1.3 with one on each: the products alone, without loads,
// splits and meetings, 0.56 and 0.8. Split between the products of both halves of a step; all in the first half, 1.06 and 1.4.
// The share of K that a block takes (gridDim.y of them) keeps the units busy where the result has few tiles; its sums then go
// to `partial` and are added by `gemm_mid_sum_kernel`.
// Measured at 401 rows on weights that no cache holds, us, by the float32 instructions (32x32x2, which this took the place of) and
// so: 8,192 columns of K 2,048 151 / 90, 6,144 of 2,048 134 / 75, 2,048 of 8,192 142 / 93, 2,048 of 2,048 46 / 33, 3,072 of 1,024
// 44 / 26, 1,024 of 1,024 17.8 / 17.0.
template <int MI, int NI, int WM, int WN>
__global__ void __launch_bounds__(64 * WM * WN)
gemm_f32_parts_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
                      const float* __restrict__ residual, void* __restrict__ out, int out_dtype, int act,
                      float* __restrict__ partial, int whole, int M, int N, int K, int tiles_m, int steps_per_share) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int T = 64 * WM * WN, TM = 32 * MI * WM, TN = 32 * NI * WN, ROWS = TM + TN;
  constexpr int PLANE = ROWS * 64, STAGE = 3 * PLANE;     // bytes: a part of a step's rows (32 of K), all three parts
  constexpr int L = ROWS * 8 / T;                         // loads of a thread a step, of T / 8 rows each
  static_assert(TM % (T / 8) == 0 && TN % (T / 8) == 0, "a load is of rows of x or of w");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int wm = (wave % WM) * 32 * MI, wn = (wave / WM) * 32 * NI;
  const int at = by_xcd(blockIdx.x, gridDim.x);
  const int m0 = at % tiles_m * TM, n0 = at / tiles_m * TN;
  const int first = blockIdx.y * steps_per_share, steps = min(K / 32 - first, steps_per_share);
  // 8 threads take the 128 bytes of a row; what a thread loads at step 0, in bytes from the tile's first row
  const int lrow = tid >> 3, lchunk = tid & 7;
  const auto xtile = __builtin_amdgcn_make_buffer_rsrc((void*)(x + (size_t)m0 * K + 32 * first), 0, -1, 0x00020000);
  const auto wtile = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)n0 * K + 32 * first), 0, -1, 0x00020000);
  int from[L];
#pragma unroll
  for (int j = 0; j < L; ++j) {
    const int row = j * (T / 8) + lrow;
    from[j] = 4 * ((j * (T / 8) < TM ? min(row, M - 1 - m0) : min(row - TM, N - 1 - n0)) * K + 4 * lchunk);
  }
  // 16-byte chunks (8 of K) of a row of 64 bytes, swizzled so that 16 rows' reads of one chunk meet no bank twice
  char* dst = smem + lrow * 64 + (((lchunk >> 1) ^ ((lrow >> 2) & 3)) * 16) + (lchunk & 1) * 8;
  f32x4 raw[3][L];
  auto load = [&](int set, int t) {
    const int k = 128 * min(t, steps - 1);
#pragma unroll
    for (int j = 0; j < L; ++j)
      raw[set][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(j * (T / 8) < TM ? xtile : wtile, from[j], k, 0));
  };
  uint2 part[L][3];
  auto split = [&](int set, int j) {
    const f32x4 v = raw[set][j];
    float r[4] = {v[0], v[1], v[2], v[3]};
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
      unsigned two[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const bf16x2 b = {(bf16_t)r[2 * e], (bf16_t)r[2 * e + 1]};
        two[e] = __builtin_bit_cast(unsigned, b);
        if (p < 2) {
          r[2 * e] -= __uint_as_float(two[e] << 16);
          r[2 * e + 1] -= __uint_as_float(two[e] & 0xffff0000u);
        }
      }
      part[j][p] = make_uint2(two[0], two[1]);
    }
  };
  auto write = [&](int stage, int j) {
#pragma unroll
    for (int p = 0; p < 3; ++p) *(uint2*)(dst + stage * STAGE + j * (T / 8) * 64 + p * PLANE) = part[j][p];
  };
  f32x16 acc[MI][NI], low[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = low[i][j][e] = 0.f;
  const int swizzle = (l32 >> 2) & 3;
  bf16x8 a[2][MI][3], b[2][NI][3];
  auto frags = [&](int stage, int s) {
    const char* base = smem + stage * STAGE + l32 * 64 + (((2 * s + half) ^ swizzle) * 16);
#pragma unroll
    for (int p = 2; p >= 0; --p) {
#pragma unroll
      for (int i = 0; i < MI; ++i) a[s][i][2 - p] = *(const bf16x8*)(base + (2 - p) * PLANE + (wm + 32 * i) * 64);
#pragma unroll
      for (int j = 0; j < NI; ++j) b[s][j][p] = *(const bf16x8*)(base + p * PLANE + (TM + wn + 32 * j) * 64);
    }
  };
  auto products = [&](int s) {
    constexpr int pa[6] = {0, 0, 1, 1, 2, 0}, pb[6] = {2, 1, 1, 0, 0, 0};
#pragma unroll
    for (int p = 0; p < 6; ++p)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          if (p < 5) low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[s][j][pb[p]], a[s][i][pa[p]], low[i][j], 0, 0, 0);
          else acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[s][j][pb[p]], a[s][i][pa[p]], acc[i][j], 0, 0, 0);
        }
  };
  load(0, 0);
  load(1, 1);
  load(2, 2);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < L; ++j) split(0, j), write(0, j);
#pragma unroll
  for (int j = L / 2; j < L; ++j) split(1, j);
  __syncthreads();
  frags(0, 0);
  // Step t (its rows in stage t % 2, the first half of its fragments in registers): the meeting is in the middle, and the next
  // step's first fragments come during the second half; the next step's rows are split beside the products of both halves.
  // (a product, and a share of the 11 instructions that two elements take to split, in turn)
  auto in_turn = [&] {
    constexpr int P = 6 * MI * NI, V = (11 * L + P - 1) / P;
#pragma unroll
    for (int i = 0; i < P; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x2, V, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto step = [&](auto place, int t) {
    constexpr int u = decltype(place)::value, stage = u & 1;
    frags(stage, 1);
    load(u % 3, t + 3);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = L / 2; j < L; ++j) write(stage ^ 1, j);
    products(0);
#pragma unroll
    for (int j = 0; j < L / 2; ++j) split((u + 1) % 3, j), write(stage ^ 1, j);
    in_turn();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    frags(stage ^ 1, 0);
    __builtin_amdgcn_sched_barrier(0);
    products(1);
#pragma unroll
    for (int j = L / 2; j < L; ++j) split((u + 2) % 3, j);
    in_turn();
  };
  int t = 0;
  for (; t + 6 <= steps; t += 6) {
    step(std::integral_constant<int, 0>{}, t);
    step(std::integral_constant<int, 1>{}, t + 1);
    step(std::integral_constant<int, 2>{}, t + 2);
    step(std::integral_constant<int, 3>{}, t + 3);
    step(std::integral_constant<int, 4>{}, t + 4);
    step(std::integral_constant<int, 5>{}, t + 5);
  }
  if (t < steps) step(std::integral_constant<int, 0>{}, t);
  if (t + 1 < steps) step(std::integral_constant<int, 1>{}, t + 1);
  if (t + 2 < steps) step(std::integral_constant<int, 2>{}, t + 2);
  if (t + 3 < steps) step(std::integral_constant<int, 3>{}, t + 3);
  if (t + 4 < steps) step(std::integral_constant<int, 4>{}, t + 4);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] += low[i][j];
  // An element that is no finite number: an operand was none, or was rounded to one (from 3.395e38 on), and its parts are no
  // sum of it. It is made again from the operands themselves.
  auto checked = [&](float v, int m, int n) {
    if (__builtin_expect(fabsf(v) <= 3.4028235e38f, 1)) return v;
    const float *xr = x + (size_t)m * K + 32 * first, *wr = w + (size_t)n * K + 32 * first;
    float sum = 0.f;
    for (int k = 0; k < 32 * steps; ++k) sum = fmaf(xr[k], wr[k], sum);
    return sum;
  };
  const int mw = m0 + wm, nw = n0 + wn;
  if (partial) {
    // A share's sums go out from the registers as they lie, four columns of a lane together (N is a multiple of 4): through LDS,
    // as the result below, the whole kernel took 1.1 us longer.
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int m = mw + 32 * i + l32;
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int n = nw + 32 * j + 8 * g + 4 * half;
          if (n >= N) continue;
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * g + e];
          const float none = (v[0] * 0.f + v[1] * 0.f) + (v[2] * 0.f + v[3] * 0.f);     // 0, or no number where one of them is not finite
          if (__builtin_expect(none != none, 0)) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = checked(v[e], m, n + e);
          }
          *(f32x4*)(partial + ((size_t)blockIdx.y * M + m) * N + n) = v;
        }
    }
    return;
  }
  __syncthreads();      // the stages are free: the result goes through them
  float added[NI][16];
#pragma unroll
  for (int j = 0; j < NI; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) added[j][e] = bias ? bias[min(nw + 32 * j + 8 * (e >> 2) + 4 * half + (e & 3), N - 1)] : 0.f;
  // (one question for all elements, as a rule none is: the way that is not taken stays out of the other's code)
  float none = 0.f;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) none += acc[i][j][e] * 0.f;
  if (__builtin_expect(none != none, 0)) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int m = mw + 32 * i + l32, n = nw + 32 * j + 8 * (e >> 2) + 4 * half + (e & 3);
          if (m < M && n < N) acc[i][j][e] = checked(acc[i][j][e], m, n);
        }
  }
  with_act(act, [&](auto activation) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = activation(acc[i][j][e] + added[j][e]);
  });
  auto value = [&](int i, int j, int e, int, int) { return acc[i][j][e]; };
  Tile<MI, NI, 2, WM, WN>::template hand_out<float, 32 * NI>(smem, value, [&](int r, int c, f32x4 chunk, int) {
    if (mw + r >= M || nw + c >= N) return;
    const size_t o = (size_t)(mw + r) * N + nw + c;
    if (whole) {
      if (residual) chunk += *(const f32x4*)(residual + o);
      *(f32x4*)((float*)out + o) = chunk;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (nw + c + e < N) store_any(out, out_dtype, o + e, chunk[e] + (residual ? residual[o + e] : 0.f));
    }
  });
}

__global__ void gemm_mid_sum_kernel(const float* __restrict__ partial, const float* __restrict__ bias,
                                    const float* __restrict__ residual, void* __restrict__ out, int out_dtype, int act, int M,
                                    int N, int shares);

// What follows a product whose K was shared out: the sum of the shares, or, with `left`, nothing but their number (1: the result
// is made); whoever asked for it adds them (`tnx_shares_norm` or `tnx_gemm_shares_sum`).
static int sum_shares(const float* partial, const float* bias, const float* residual, void* out, int out_dtype, int act, int M, int N,
                      int shares, int* left, hipStream_t stream) {
  if (left) *left = shares;
  if (shares > 1 && !left) {
    gemm_mid_sum_kernel<<<(unsigned)(((size_t)M * N / 4 + 255) / 256), 256, 0, stream>>>(partial, bias, residual, out, out_dtype,
                                                                                        act, M, N, shares);
    TNX_CHECK_LAUNCH("gemm_mid_sum");
  }
  return 0;
}

// The sum alone, of a product that left its shares.
extern "C" int tnx_gemm_shares_sum(const float* partial, const float* bias, const float* residual, float* out, int M, int N, int shares,
                                   hipStream_t stream) {
  TNX_REQUIRE(M > 0 && N > 0 && N % 4 == 0 && shares > 1 && partial && out && ((uintptr_t)partial & 15) == 0, "gemm_shares_sum: bad sizes");
  return sum_shares(partial, bias, residual, out, TNX_F32, TNX_ACT_NONE, M, N, shares, nullptr, stream);
}


template <int MI, int NI, int WM, int WN>
static int launch_f32_parts(const float* x, const float* w, const float* bias, const float* residual, void* out, int out_dtype,
                            int act, float* partial, int M, int N, int K, int shares, int* left, hipStream_t stream) {
  constexpr int bytes = 2 * 3 * (32 * MI * WM + 32 * NI * WN) * 64;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_f32_parts_kernel<MI, NI, WM, WN>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    TNX_REQUIRE(e == hipSuccess, "gemm_f32: cannot reserve %d bytes of LDS: %s", bytes, hipGetErrorString(e));
    configured = true;
  }
  const int tiles_m = (M + 32 * MI * WM - 1) / (32 * MI * WM), tiles_n = (N + 32 * NI * WN - 1) / (32 * NI * WN);
  const int per = (K / 32 + shares - 1) / shares;
  shares = (K / 32 + per - 1) / per;
  // whole chunks of 16 bytes in every row of the result
  const int whole = N % 4 == 0 && out_dtype == TNX_F32 && ((uintptr_t)out | (uintptr_t)residual) % 16 == 0;
  gemm_f32_parts_kernel<MI, NI, WM, WN><<<dim3(tiles_m * tiles_n, shares), 64 * WM * WN, bytes, stream>>>(
      x, w, bias, residual, out, out_dtype, act, shares > 1 ? partial : nullptr, whole, M, N, K, tiles_m, per);
  TNX_CHECK_LAUNCH("gemm_f32_parts");
  return sum_shares(partial, bias, residual, out, out_dtype, act, M, N, shares, left, stream);
}

// The most floats that the shares' sums of one product may take (32 MB).
constexpr long long F32_SHARES_MOST = 8 << 20;

// The tile (128 x 128, 64 x 128, 64 x 64) and the shares of K, by what a launch takes in us: a step of 32 of K of the blocks that
// the fullest compute unit has (measured: one of 128 x 128 1.28, and no second fits its LDS; 64 x 128 0.70 and 1.35 for one and two
// at once; 64 x 64 0.50, 0.88, 1.26), a beginning and an end, and the sum of the shares.
// Up to 128 rows the launch is a chain of few steps, and its parts are a fit to 2,253 launches: 17 matrices from 64 x 64 to 12,288 x
// 4,096, 17 to 128 rows, all tiles, up to 16 shares of two steps or more, on weights that no cache holds; what it picks takes 1.01 of
// the quickest on average, 1.14 at most. Beyond, up to eight shares of four steps: fewer of them would be up to 15 % quicker at 180
// to 400 rows of many columns, at sums of twice the length and error.
// us by the float32 instructions (32x32x2) before / so: 1,024 x 1,024 at 17, 64 and 256 rows 8.7 / 8.7, 9.4 / 9.4, 13.3 / 14.5; 3,072 x 1,024
// at 17 and 64 10.6 / 10.7, 12.3 / 12.8; 1,024 x 4,096 15.9 / 12.3 and 16.7 / 14.0; 2,048 x 2,048 at 64 13.5 / 14.0; the worst 2,304 x 768 at
// 17 and 64, 8.8 / 9.4 and 10.4 / 11.0, and single tiles (64 x 64 of K 64 5.6 / 6.0): the split of an operand is a longer beginning.
static void choose_f32_tiles(int M, int N, int K, int& tile, int& shares) {
  const int units = tnx_compute_units(), steps = K / 32, few = M <= 128;
  const int sizes[3][2] = {{128, 128}, {64, 128}, {64, 64}};
  const double block_step[2][3] = {{1.28, 0.65, 0.38}, {1.0, 0.655, 0.346}}, step_more[2][3] = {{0.0, 0.05, 0.12}, {0.0, 0.0, 0.19}};
  const double ends[2][3] = {{0.0, 8.0, 8.0}, {6.1, 5.1, 5.5}}, block_ends[2][3] = {{8.0, 0.0, 0.0}, {0.45, 0.66, 0.0}};
  const double sum[2] = {5.0, 1.0}, sum_element[2] = {1e-6, 2e-6};
  double best = 1e30;
  for (int i = 0; i < 3; ++i) {
    const long long tiles = (long long)((M + sizes[i][0] - 1) / sizes[i][0]) * ((N + sizes[i][1] - 1) / sizes[i][1]);
    for (int s = 1; s <= (few ? 16 : 8) && (s == 1 || (N % 4 == 0 && steps / s >= (few ? 2 : 4) && (long long)s * M * N <= F32_SHARES_MOST)); ++s) {
      const int per = (steps + s - 1) / s;
      const long long blocks = (tiles * (few ? (steps + per - 1) / per : s) + units - 1) / units;
      double cost = per * ((double)blocks * block_step[few][i] + step_more[few][i]) + ends[few][i] + blocks * block_ends[few][i];
      if (s > 1) cost += sum[few] + (double)M * N * (s + 1) * sum_element[few];
      if (cost < best) best = cost, tile = i, shares = s;
    }
  }
}

// How many floats of workspace `tnx_gemm_f32` wants for a product: those of the shares' sums, 0 where K is not shared out.
extern "C" int tnx_gemm_f32_workspace(int M, int N, int K) {
  if (M <= 16 || N <= 0 || K < 32 || K % 32 != 0) return 0;
  int tile = 0, shares = 1;
  choose_f32_tiles(M, N, K, tile, shares);
  return shares > 1 ? shares * M * N : 0;
}

// `tile` as in `choose_f32_tiles`.
static int f32_parts(const float* x, const float* w, const float* bias, const float* residual, void* out, int out_dtype, int act, int M,
                     int N, int K, int tile, int shares, float* workspace, int* left, hipStream_t stream) {
#define F32_TILES(MI, NI, WM, WN) \
  launch_f32_parts<MI, NI, WM, WN>(x, w, bias, residual, out, out_dtype, act, workspace, M, N, K, shares, left, stream)
  return tile == 0 ? F32_TILES(1, 2, 4, 2) : tile == 1 ? F32_TILES(1, 1, 2, 4) : F32_TILES(1, 1, 2, 2);
#undef F32_TILES
}

// The product by parts with a tile and shares of the caller's (`tnx_gemm_f32` chooses them).
extern "C" int tnx_gemm_f32_parts(const float* x, const float* w, const float* bias, const float* residual, void* out, int out_dtype,
                                  int act, int M, int N, int K, int tile, int shares, float* workspace, size_t workspace_floats,
                                  hipStream_t stream) {
  TNX_REQUIRE(M > 0 && N > 0 && K > 0 && K % 32 == 0 && K < 1 << 22 && ((uintptr_t)x | (uintptr_t)w | (uintptr_t)workspace) % 16 == 0,
              "gemm_f32_parts: K in 32s below 2^22 and operands 16-byte aligned, got M=%d N=%d K=%d", M, N, K);
  TNX_REQUIRE(tile >= 0 && tile <= 2 && shares >= 1 && shares <= 16 && shares <= K / 32, "gemm_f32_parts: tile 0 to 2, up to 16 shares");
  TNX_REQUIRE(shares == 1 || (N % 4 == 0 && workspace && workspace_floats >= (size_t)shares * M * N),
              "gemm_f32_parts: shares want N a multiple of 4 and a workspace of shares x M x N floats");
  return f32_parts(x, w, bias, residual, out, out_dtype, act, M, N, K, tile, shares, workspace, nullptr, stream);
}

// `workspace`: as many floats as `tnx_gemm_f32_workspace` names for the sizes; with less, K is not shared out.
static int gemm_f32(const float* x, const float* w, const float* bias, const float* residual, void* out, int out_dtype, int act,
                    int M, int N, int K, float* workspace, size_t workspace_floats, int* left, hipStream_t stream) {
  if (left) *left = 1;
  TNX_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  if (M == 0) return 0;
  if (M <= 16 && K % 4 == 0 && ((uintptr_t)x | (uintptr_t)w) % 16 == 0) {
    f32_skinny(x, w, bias, residual, out, out_dtype, act, M, N, K, NoScatter{}, stream);
    TNX_CHECK_LAUNCH("gemm_f32_skinny");
    return 0;
  }
  if (K % 32 == 0 && K < 1 << 22 && ((uintptr_t)x | (uintptr_t)w | (uintptr_t)workspace) % 16 == 0) {
    int tile = 0, shares = 1;
    choose_f32_tiles(M, N, K, tile, shares);
    if (shares > 1 && (workspace == nullptr || workspace_floats < (size_t)shares * M * N)) shares = 1;
    return f32_parts(x, w, bias, residual, out, out_dtype, act, M, N, K, tile, shares, workspace, left, stream);
  }
  dim3 grid((N + F32_TILE - 1) / F32_TILE, (M + F32_TILE - 1) / F32_TILE);
  TNX_REQUIRE(grid.y <= 65535, "gemm_f32: M=%d is too large", M);
  gemm_f32_kernel<<<grid, 256, 0, stream>>>(x, w, bias, residual, out, out_dtype, act, M, N, K);
  TNX_CHECK_LAUNCH("gemm_f32");
  return 0;
}

extern "C" int tnx_gemm_f32(const float* x, const float* w, const float* bias, const float* residual, void* out,
                            int out_dtype, int act, int M, int N, int K, float* workspace, size_t workspace_floats,
                            hipStream_t stream) {
  return gemm_f32(x, w, bias, residual, out, out_dtype, act, M, N, K, workspace, workspace_floats, nullptr, stream);
}

// ------------------------------------------------------------------------------------------ bfloat16, tiled

#define BT_M 128
#define BT_N 128
#define BT_K 32
#define BT_STRIDE 40  // elements per staged row: 32 of data, 8 of padding against LDS bank conflicts

template <bool QKV>
__global__ void __launch_bounds__(256)
gemm_bf16_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const float* __restrict__ bias,
                 const float* __restrict__ residual, void* __restrict__ out, int out_dtype, int act, int M, int N,
                 int K, QkvScatter sc) {
  __shared__ __attribute__((aligned(16))) bf16_t xs[BT_M * BT_STRIDE];
  __shared__ __attribute__((aligned(16))) bf16_t ws[BT_N * BT_STRIDE];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 64, wn = (wave >> 1) * 64;
  const int m0 = blockIdx.y * BT_M, n0 = blockIdx.x * BT_N;
  const int l32 = lane & 31, lhalf = lane >> 5;

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  bf16x8 rx[2], rw[2];
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  // No load depends on a branch: rows beyond M or N read the last row, a step beyond K reads the last
  // whole chunk of the row, and what must count as zero is zeroed after the load.
  const bf16_t* xsrc[2];
  const bf16_t* wsrc[2];
  int kofs[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int c = tid + 256 * j;
    const int row = c >> 2;
    kofs[j] = (c & 3) * 8;
    xsrc[j] = x + (size_t)min(m0 + row, M - 1) * K;
    wsrc[j] = w + (size_t)min(n0 + row, N - 1) * K;
  }
  auto fetch = [&](int k0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int k = k0 + kofs[j];
      const bool k_ok = k + 8 <= K;
      const int kc = k_ok ? k : K - 8;
      const bf16x8 xv = *(const bf16x8*)(xsrc[j] + kc);
      const bf16x8 wv = *(const bf16x8*)(wsrc[j] + kc);
      rx[j] = k_ok ? xv : zero;
      rw[j] = k_ok ? wv : zero;
    }
  };
  fetch(0);
  for (int k0 = 0; k0 < K; k0 += BT_K) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int c = tid + 256 * j;
      const int row = c >> 2, kc = (c & 3) * 8;
      *(bf16x8*)(xs + row * BT_STRIDE + kc) = rx[j];
      *(bf16x8*)(ws + row * BT_STRIDE + kc) = rw[j];
    }
    __syncthreads();
    if (k0 + BT_K < K) fetch(k0 + BT_K);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = *(const bf16x8*)(xs + (wm + i * 32 + l32) * BT_STRIDE + ks * 16 + lhalf * 8);
#pragma unroll
      for (int j = 0; j < 2; ++j) b[j] = *(const bf16x8*)(ws + (wn + j * 32 + l32) * BT_STRIDE + ks * 16 + lhalf * 8);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  }
  // acc[i][j][e] is row 8*(e/4) + 4*(lane/32) + e%4, column lane%32 of its 32x32 tile.
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + wn + j * 32 + l32;
      if (n >= N) continue;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm + i * 32 + 8 * (e >> 2) + 4 * lhalf + (e & 3);
        if (m < M) {
          if (QKV) {
            // (the element beside this one is the neighbouring lane's: N is even, so both are there or neither)
            const float v = acc[i][j][e] + (bias ? bias[n] : 0.f);
            qkv_store(v, lane_dpp<TNX_DPP_XOR1>(v), m, n, sc, sc.token_page[m], sc.token_off[m]);
          } else {
            epilogue_store(acc[i][j][e], m, n, N, bias, residual, out, out_dtype, act);
          }
        }
      }
    }
}

// ------------------------------------------------------------------------------------------ bfloat16, wide tiles

#define WT_M 256
#define WT_N 256
typedef __attribute__((address_space(3))) void* lds_ptr;
typedef const __attribute__((address_space(1))) void* glb_ptr;

// out[M][N] = x[M][K] w[N][K]^T. Tiles of 64 MI x 256 x BK (MI 4: 256 rows, MI 2: 128 rows, for results too
// narrow to give every compute unit a tile of 256), four waves (2 x 2), each 32 MI x 128 of the result as
// MI x 4 MFMA 32x32x16 tiles (64 MI accumulator registers; a fragment read from LDS serves four products).
// Operand tiles go from global memory straight into LDS, NSTAGE stages deep, 16-byte chunks swizzled by row
// so that the fragment reads are free of bank conflicts (the banks repeat every 256 bytes).
// The depth of a step and the number of stages the launcher uses: 64 deep, two stages (all of LDS for the
// larger tile). 32 deep with three or four stages, so that a tile's loads have two steps to land, measured
// 6 to 18% slower at 2,048 to 8,192 rows.
constexpr int WIDE_BK = 64, WIDE_NSTAGE = 2;
template <int BK, int NSTAGE, int MI>
__global__ void __launch_bounds__(256, 1)
gemm_bf16_wide_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const float* __restrict__ bias,
                const float* __restrict__ residual, void* __restrict__ out, int out_dtype, int act, int M, int N,
                int K, int tiles_m, int tiles_n) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int CPR = BK / 8;                     // 16-byte chunks a row
  constexpr int ROWB = BK * 2;                    // bytes a row
  constexpr int TM = 64 * MI;                     // rows of x a tile takes
  constexpr int STAGE = (TM + WT_N) * ROWB;       // bytes of one stage
  constexpr int RPI = 64 / CPR;                   // rows a wave's load instruction covers
  constexpr int LPA = TM / (4 * RPI);             // load instructions a wave issues for a tile of x
  constexpr int LPT = WT_N / (4 * RPI);           // and of w
  constexpr int KS = BK / 16;                     // k16 steps
  // the k16 steps of a tile between whose products the next tile's loads are issued: the first two, so that the
  // last load has half a tile's time to land before the barrier (over all four: 3 to 8% slower; in the first: 2%)
  constexpr int LOAD_STEPS = KS < 2 ? KS : 2;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave & 1) * 32 * MI, wn = (wave >> 1) * 128;
  const int nb = tiles_m * tiles_n;
  int bid = blockIdx.x;
  if (nb % 8 == 0) bid = (bid & 7) * (nb >> 3) + (bid >> 3);
  const int tm = bid % tiles_m, tn = bid / tiles_m;
  const int m0 = tm * TM, n0 = tn * WT_N;
  const int l32 = lane & 31, lhalf = lane >> 5;

  f32x16 acc[MI][4];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // 16 lanes are served a cycle and the banks repeat every 256 bytes: 16 consecutive rows must put the chunk
  // they read into 16 different 16-byte places of those 256 bytes
  auto swz = [&](int row) { return CPR == 8 ? ((row >> 1) & 7) : ((row >> 2) & 3); };
  const int lrow = lane / CPR, lpos = lane % CPR;
  const bf16_t* xsrc[LPA];
  const bf16_t* wsrc[LPT];
#pragma unroll
  for (int j = 0; j < LPA; ++j) {
    const int row = (LPA * wave + j) * RPI + lrow;
    xsrc[j] = x + (size_t)min(m0 + row, M - 1) * K + 8 * (lpos ^ swz(row));
  }
#pragma unroll
  for (int j = 0; j < LPT; ++j) {
    const int row = (LPT * wave + j) * RPI + lrow;
    wsrc[j] = w + (size_t)min(n0 + row, N - 1) * K + 8 * (lpos ^ swz(row));
  }
  auto issue_part = [&](int stage, int k0, int part, int parts) {      // loads part, part + parts, ... of a tile
    char* a_dst = smem + stage * STAGE + (LPA * wave) * 1024;
    char* b_dst = smem + stage * STAGE + TM * ROWB + (LPT * wave) * 1024;
#pragma unroll
    for (int j = 0; j < LPA; ++j)
      if (j % parts == part)
        load_to_lds(xsrc[j] + k0, lds_offset(a_dst + j * 1024));
#pragma unroll
    for (int j = 0; j < LPT; ++j)
      if (j % parts == part)
        load_to_lds(wsrc[j] + k0, lds_offset(b_dst + j * 1024));
  };
  auto issue = [&](int stage, int k0) { issue_part(stage, k0, 0, 1); };
  int a_off[MI], b_off[4];
#pragma unroll
  for (int i = 0; i < MI; ++i) a_off[i] = (wm + 32 * i + l32) * ROWB;
#pragma unroll
  for (int j = 0; j < 4; ++j) b_off[j] = TM * ROWB + (wn + 32 * j + l32) * ROWB;
  const int rsw = swz(l32);

  const int steps = K / BK;
#pragma unroll
  for (int p = 0; p < NSTAGE - 1; ++p)
    if (p < steps) issue(p, p * BK);
  constexpr int AHEAD = 1;                        // k16 steps between asking for fragments and using them (2: 3% slower)
  bf16x8 a[AHEAD + 1][MI], b[AHEAD + 1][4];
  auto frags = [&](int slot, const char* base, int s) {
    const int coff = ((2 * s + lhalf) ^ rsw) * 16;
#pragma unroll
    for (int i = 0; i < MI; ++i) a[slot][i] = *(const bf16x8*)(base + a_off[i] + coff);
#pragma unroll
    for (int j = 0; j < 4; ++j) b[slot][j] = *(const bf16x8*)(base + b_off[j] + coff);
  };
  auto products = [&](int slot) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[slot][j], a[slot][i], acc[i][j], 0, 0, 0);
  };
  int stage = 0;
  auto iteration = [&](int t, auto with_loads) {
    constexpr bool more = decltype(with_loads)::value;
    // tile t has landed when at most the loads of the NSTAGE - 2 tiles after it are still in flight
    const int ahead = min(NSTAGE - 2, steps - 1 - t);
    if (ahead >= 2) __builtin_amdgcn_s_waitcnt(0x0F70 | ((2 * (LPA + LPT)) & 15) | (((2 * (LPA + LPT)) >> 4) << 14));
    else if (ahead == 1) __builtin_amdgcn_s_waitcnt(0x0F70 | ((LPA + LPT) & 15) | (((LPA + LPT) >> 4) << 14));
    else __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    // the stage that tile t - 1 was read from is free now: tile t + NSTAGE - 1 goes there, its loads spread
    // over this tile's steps between the products
    const int nstage = (stage + NSTAGE - 1) % NSTAGE, nk = (t + NSTAGE - 1) * BK;
    const char* base = smem + stage * STAGE;
    frags(0, base, 0);
    if (AHEAD == 2 && KS > 1) frags(1, base, 1);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      // the fragments of the step after next are asked for first, in one run; this step's products run
      // while they arrive
      if (s + AHEAD < KS) frags((s + AHEAD) % (AHEAD + 1), base, s + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
      if (more && s < LOAD_STEPS) {
        issue_part(nstage, nk, s, LOAD_STEPS);
        products(s % (AHEAD + 1));
#pragma unroll
        for (int g = 0; g < (LPA + LPT) / LOAD_STEPS; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x008, 4 * MI * LOAD_STEPS / (LPA + LPT), 0);
          __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
      } else {
        products(s % (AHEAD + 1));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    stage = stage + 1 == NSTAGE ? 0 : stage + 1;
  };
  int t = 0;
  for (; t + NSTAGE - 1 < steps; ++t) iteration(t, std::true_type{});
  for (; t < steps; ++t) iteration(t, std::false_type{});
  // acc[i][j][e] of a lane is out[m][n] at m = 32 i + lane % 32, n = 32 j + 8 (e / 4) + 4 (lane / 32) + e % 4 of the
  // wave's 32 MI x 128: four consecutive n a register group. A block of 32 rows at a time goes through LDS (the
  // stages are free now), so that rows are written to memory 16 bytes a lane, whole lines at a time.
  __syncthreads();
  const bool relu = act == TNX_ACT_RELU;
  const bool wide = out_dtype == TNX_F32;
  const int esz = wide ? 4 : 2;
  const int rowb = 128 * esz + 16;                     // bytes of a staged row, padded against bank conflicts
  char* mine = smem + wave * (32 * (128 * 4 + 16));
#pragma unroll
  for (int i = 0; i < MI; ++i) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int nl = 32 * j + 8 * q + 4 * lhalf;     // first of this lane's four columns within the wave's 128
        const int n = n0 + wn + nl;
        float v[4];
        f32x4 bv = {0.f, 0.f, 0.f, 0.f};
        if (bias) bv = *(const f32x4*)(bias + min(n, N - 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = acc[i][j][4 * q + e] + bv[e];
          if (relu) v[e] = fmaxf(v[e], 0.f);
        }
        char* dst = mine + l32 * rowb + nl * esz;
        if (wide) {
          *(f32x4*)dst = (f32x4){v[0], v[1], v[2], v[3]};
        } else {
          bf16x4 pk = {(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
          *(bf16x4*)dst = pk;
        }
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // read back: a row of 128 outputs is 16 (bfloat16) or 32 (float32) chunks of 16 bytes
    const int cpr_out = 128 * esz / 16;
    const int rows_pass = 64 / cpr_out;
    for (int r0 = 0; r0 < 32; r0 += rows_pass) {
      const int r = r0 + lane / cpr_out, c = lane % cpr_out;
      const int m = m0 + wm + 32 * i + r;
      const int n = n0 + wn + c * (16 / esz);
      f32x4 raw = *(const f32x4*)(mine + r * rowb + c * 16);
      if (m < M && n < N) {          // N is a multiple of 8 here: a chunk is inside or outside as a whole
        const size_t idx = (size_t)m * N + n;
        if (wide) {
          if (residual) {
            const f32x4 rv = *(const f32x4*)(residual + idx);
            raw += rv;
          }
          *(f32x4*)((float*)out + idx) = raw;
        } else {
          *(f32x4*)((bf16_t*)out + idx) = raw;
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}


// Where the wide-tile kernel can stand in: whole chunks of 16 bytes in every row of the result, K in steps of 64,
// a residual only beside a float32 result, and enough rows to fill its tiles.
static bool wide_tiles_fit(int M, int N, int K, const float* residual, int out_dtype, int act) {
  return M >= 128 && K % 64 == 0 && N % 8 == 0 && (residual == nullptr || out_dtype == TNX_F32) &&
         (act == TNX_ACT_NONE || act == TNX_ACT_RELU);
}

template <int MI>
static int launch_wide_tiles(const bf16_t* x, const bf16_t* w, const float* bias, const float* residual, void* out,
                             int out_dtype, int act, int M, int N, int K, hipStream_t stream) {
  constexpr int TM = 64 * MI;
  const int tiles_m = (M + TM - 1) / TM, tiles_n = (N + WT_N - 1) / WT_N;
  constexpr int bytes = WIDE_NSTAGE * (TM + WT_N) * WIDE_BK * 2;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_bf16_wide_kernel<WIDE_BK, WIDE_NSTAGE, MI>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) {
      tnx_set_error("gemm_bf16: cannot reserve %d bytes of LDS: %s", bytes, hipGetErrorString(e));
      return 2;
    }
    configured = true;
  }
  gemm_bf16_wide_kernel<WIDE_BK, WIDE_NSTAGE, MI><<<tiles_m * tiles_n, 256, bytes, stream>>>(x, w, bias, residual, out, out_dtype,
                                                                             act, M, N, K, tiles_m, tiles_n);
  return 0;
}

static int launch_wide(const bf16_t* x, const bf16_t* w, const float* bias, const float* residual, void* out,
                       int out_dtype, int act, int M, int N, int K, hipStream_t stream) {
  // tiles of 256 rows where they give (nearly) every compute unit one, tiles of 128 rows otherwise
  const int full = ((M + 255) / 256) * ((N + WT_N - 1) / WT_N);
  if (full >= 200) return launch_wide_tiles<4>(x, w, bias, residual, out, out_dtype, act, M, N, K, stream);
  return launch_wide_tiles<2>(x, w, bias, residual, out, out_dtype, act, M, N, K, stream);
}

// ------------------------------------------------------------------------------------------ bfloat16, few rows

// Products of few rows next to a norm: a block asks for the rows and then for its first weights, and norms the rows while the
// weights come: all of them into LDS as the operand (NORM_OPERAND), or their means and deviations alone, with which a thread
// norms the element of the residual that it adds (NORM_RESIDUAL: behind a sum, what a norm gives is the stream itself, operand of
// the next product and residual of the one after that). The rows come first because loads are waited for in the order they were
// made: asked for after the weights they made every product 2 us longer. Statistics in float32 in two passes over registers, as
// the norm's own kernel takes them; the operand is read from LDS, which is nearer than rows that other units left in memory.
// Measured, us, at 1 and 8 rows: the norm's kernel and the product / the norm folded into the product (`NormFold`) / so:
// 4,096 columns of K 1,024 6.4, 7.0 / 5.2, 6.4 / 4.2, 4.5; 8,192 of 2,048 11.6, 12.3 / 9.9, 11.8 / 9.2, 10.1; 10,240 of 2,560 15.4, 16.3 /
// 14.3, 16.0 / 13.5, 15.3; but 16,384 of 4,096 28.5, 29.6 / 27.3, 30.5 / 28.8, 32.3: wider rows take the registers and the time
// of too many blocks. As a residual of 1,024, with the product of K 1,024 and of 4,096: 3.4, 4.0 and 6.1, 7.3 with the normed
// residual there, 3.8, 4.4 and 6.4, 7.9 so. Norm, first product and second with the residual of a feed-forward of four times the
// width, at 1 and 8 rows: 1,024 12.1, 13.8 / 10.7, 12.4; 1,536 17.8, 19.6 / 16.3, 19.2; 2,048 22.5, 25.6 / 21.1, 24.9, where it ends.
struct RowNorm {
  const float* x;        // [M][width] float32
  const float* weight;   // [width], with `bias` or both null
  const float* bias;
  float eps;
  int center;            // 0: a norm that only scales
};
enum NormKind { NORM_NONE = 0, NORM_OPERAND = 1, NORM_RESIDUAL = 2 };
struct NoNorm {};
template <int KIND>
using NormArg = std::conditional_t<KIND == NORM_NONE, NoNorm, RowNorm>;
constexpr int NORM_OPERAND_WIDTH = 3072, NORM_RESIDUAL_WIDTH = 2048;

// Rows wave, wave + 4 (below M) of the norm's by this wave of four. `ask` comes before the block asks for its weights: loads are
// waited for in the order they were made.
template <int ROWS, int PER, bool OPERAND>
struct NormedRows {
  f32x4 v[ROWS][PER], gw[OPERAND ? PER : 1], gb[OPERAND ? PER : 1];
  __device__ __forceinline__ void ask(const RowNorm& n, int M, int width) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int j = 0; j < PER; ++j)
        if (256 * j < width) v[r][j] = *(const f32x4*)(n.x + (size_t)min(wave + 4 * r, M - 1) * width + min(256 * j + 4 * lane, width - 4));
    if constexpr (OPERAND) {
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const int i = min(256 * j + 4 * lane, width - 4);
        gw[j] = n.weight ? *(const f32x4*)(n.weight + i) : (f32x4){1.f, 1.f, 1.f, 1.f};
        gb[j] = n.bias ? *(const f32x4*)(n.bias + i) : (f32x4){0.f, 0.f, 0.f, 0.f};
      }
    }
  }
  // Mean and 1 / deviation into `stat`; as the operand, the normed rows into `rows` (LDS, `pitch` elements a row).
  __device__ __forceinline__ void finish(const RowNorm& n, int M, int width, bf16_t* rows, int pitch, float (*stat)[2]) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const int m = wave + 4 * r;
      if (m >= M) continue;
      float s = 0.f, q = 0.f;
#pragma unroll
      for (int j = 0; j < PER; ++j)
        if (256 * j + 4 * lane < width) s += (v[r][j].x + v[r][j].y) + (v[r][j].z + v[r][j].w);
      const float mean = n.center ? wave_sum(s) / (float)width : 0.f;
#pragma unroll
      for (int j = 0; j < PER; ++j)
        if (256 * j + 4 * lane < width) {
          const f32x4 d = v[r][j] - mean;
          q += (d.x * d.x + d.y * d.y) + (d.z * d.z + d.w * d.w);
        }
      const float rstd = rsqrtf(wave_sum(q) / (float)width + n.eps);
      if (lane == 0) stat[m][0] = mean, stat[m][1] = rstd;
      if constexpr (OPERAND) {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
          const int i = 256 * j + 4 * lane;
          if (i >= width) continue;
          const f32x4 y = (v[r][j] - mean) * rstd * gw[j] + gb[j];
          bf16x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = (bf16_t)y[e];
          *(bf16x4*)(rows + m * pitch + i) = o;
        }
      }
    }
  }
};

// One block of WAVES waves makes 16 * RT columns of the output (RT tiles of 16 rows of `w`) for all
// M <= 16 * MT rows of `x`; with RT = 2 every fragment of `x` serves two products, which pays for wide
// matrices (N >= 16,384: 29.2 -> 27.2 us at 8 rows, 34.1 -> 29.6 at 16) and costs blocks for narrow ones.
// The waves share the K axis in steps of 128; inside a step each of the four loads of a wave covers 64
// contiguous bytes of each of its 16 weight rows (the four lane groups side by side), and `x` is read the
// same way. The weight is fetched two steps ahead of its use, `x` one step. No load in the main loop
// is conditional: rows beyond N or M and steps beyond K read a valid address and their products are
// dropped, so the compiler can keep many loads in flight. What is left of K after the last whole step of
// 128 (K % 128, a multiple of 8) is done by wave 0 with guarded loads. The partial sums of the waves meet
// in LDS.
// With SHUF the weight is read from a copy laid out for this kernel: [N/16][K/128][4][16 rows][4][8], that is
// tile after tile in the order the loads take it, so that a block streams one contiguous run of memory and
// each load of a wave covers 1 KB of it (N a multiple of 16, K of 128).
// With NORMED the rows of `x` are those of a LayerNorm's float32 input and the product is that of the
// normalised rows, without a kernel for the norm: with W' = W diag(gamma), c = W' 1 and d = W beta,
//     W (gamma (x - mean) rstd + beta) = rstd (W' (x - x0) - (mean - x0) c) + d
// for any x0. The block's waves read every element of the rows between them anyway (they share K), so the sums
// of x - x0 and of its square cost no load; x0 is the median of three elements of the row (one of them may be
// an outlier), so that what is rounded to bfloat16 for the products is small where the row has a large common
// part. `w` is W' here (tile order), `nf.c`
// and `nf.d` come with it; K is a multiple of 128.
struct NormFold {
  const float* x;      // [M][K] float32
  const float* c;      // [N]
  const float* d;      // [N]
  float eps;
  int center;          // 0: a norm that only scales (the mean is taken as 0, and nothing is shifted before rounding)
};

// With GATED the rows of `w` are gate rows and as many up rows (N of both): a block takes a tile of either, sixteen columns of
// act(gate) * up, which goes out in bfloat16 (`limit`: of the clamped form). A launch less: us, 8 rows, 4,096 gate rows of 2,048
// 11.6 / 8.9, 8,192 of 4,096 28.1 / 25.1 (`HipOps._gated_way`).
// With PAIRS the residual is the sum of `residual` and of each row's `top` (up to four) rows of `pairs`, in their order: what a mixture
// of experts leaves, whose launch for that sum takes 4 us of its own (a step of 4 such layers 446 us with it, 434 without).
template <int MT, int WAVES, bool QKV, bool SHUF, int RT, bool NORMED = false, int NORM = NORM_NONE, int ROWS = 1, int PER = 1, bool GATED = false, bool PAIRS = false>
__global__ void __launch_bounds__(WAVES * 64)
gemm_bf16_skinny_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const float* __restrict__ bias,
                        const float* __restrict__ residual, void* __restrict__ out, int out_dtype, int act, int M,
                        int N, int K, QkvScatter sc, NormFold nf, NormArg<NORM> norm, float limit = 0.f,
                        const float* __restrict__ pairs = nullptr, int top = 0) {
  static_assert(!GATED || (RT == 2 && SHUF && !QKV && !NORMED && NORM == NORM_NONE), "a tile of gate rows and one of up rows");
  static_assert(NORM == NORM_NONE || (MT == 1 && WAVES == 4 && !NORMED), "two rows a wave of four");
  __shared__ float norm_stat[NORM ? 16 : 1][2];
  extern __shared__ __attribute__((aligned(16))) char normed_rows[];
  const int norm_pitch = K + 8;       // (16 bytes more than a row: rows would share their banks)
  __shared__ float red[WAVES][MT][RT][4][64];
  __shared__ float stat[WAVES][MT][2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16 * RT;     // RT tiles of 16 weight rows a block; tile j begins at n0 + 16 j
  // element offset of the load of step s at K offset kc: W_STEP * kc + W_LOAD * s from wrow
  constexpr int W_STEP = SHUF ? 16 : 1, W_LOAD = SHUF ? 512 : 32;
  const bf16_t* wrow[RT];
#pragma unroll
  for (int j = 0; j < RT; ++j)
    wrow[j] = SHUF ? w + (size_t)(GATED ? (int)blockIdx.x + j * (N / 32) : min((int)blockIdx.x * RT + j, N / 16 - 1)) * 16 * K + (r * 4 + g) * 8
                   : w + (size_t)min(n0 + 16 * j + r, N - 1) * K + 8 * g;
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  NormedRows<ROWS, PER, NORM == NORM_OPERAND> normed;
  if constexpr (NORM != NORM_NONE) {
    normed.ask(norm, M, NORM == NORM_OPERAND ? K : N);
    __builtin_amdgcn_sched_barrier(0);
  }
  // What the end of the kernel adds (bias, residual, the folded norm's vectors) is asked for first: there it would be one
  // more time to reach memory after the last product. A thread's element q is (row, column) of `place(q)`.
  constexpr int OUTS = MT * RT * 4 / WAVES;      // elements a thread makes: MT RT tiles of 256 by 64 WAVES threads
  auto place = [&](int q, int& m, int& n) {
    const int idx = tid + q * WAVES * 64, l = idx & 63, i = (idx >> 6) & 3, j = (idx >> 8) % RT, t = idx / (256 * RT);
    m = t * 16 + (l & 15);
    n = n0 + 16 * j + 4 * (l >> 4) + i;
  };
  constexpr bool EARLY = OUTS >= 1 && OUTS <= 4 && MT * RT * 4 % WAVES == 0;
  float add[EARLY ? OUTS : 1], onto[EARLY ? OUTS : 1], fold_c[EARLY ? OUTS : 1], fold_d[EARLY ? OUTS : 1];
  float onto_w[EARLY ? OUTS : 1], onto_b[EARLY ? OUTS : 1], of_pair[PAIRS ? OUTS : 1][4];
  static_assert(!PAIRS || EARLY, "the pairs' rows are asked for before the products");
  int page[EARLY ? OUTS : 1], off[EARLY ? OUTS : 1];
  static_assert(NORM == NORM_NONE || EARLY, "the residual is normed where it was asked for");
  if constexpr (EARLY) {
#pragma unroll
    for (int q = 0; q < OUTS; ++q) {
      int m, n;
      place(q, m, n);
      m = min(m, M - 1), n = min(n, N - 1);
      add[q] = bias ? bias[n] : 0.f;
      if (NORMED) fold_c[q] = nf.c[n], fold_d[q] = nf.d[n];
      onto[q] = !QKV && residual ? residual[(size_t)m * N + n] : 0.f;
      if constexpr (PAIRS) {
#pragma unroll
        for (int c = 0; c < 4; ++c) of_pair[q][c] = pairs[((size_t)m * top + min(c, top - 1)) * N + n];
      }
      if constexpr (NORM == NORM_RESIDUAL) {
        onto[q] = norm.x[(size_t)m * N + n];
        onto_w[q] = norm.weight ? norm.weight[n] : 1.f;
        onto_b[q] = norm.bias ? norm.bias[n] : 0.f;
      }
      if (QKV) page[q] = sc.token_page[m], off[q] = sc.token_off[m];
    }
  }
  f32x4 acc[MT][RT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int j = 0; j < RT; ++j) acc[t][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const bf16_t* xrow[MT];
  const float* xfrow[MT];
  float x0[MT], s1[MT], s2[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const size_t row = (size_t)min(t * 16 + r, M - 1) * K;
    xrow[t] = NORMED || NORM == NORM_OPERAND ? nullptr : x + row + 8 * g;
    xfrow[t] = NORMED ? nf.x + row + 8 * g : nullptr;
    if (NORMED && nf.center) {
      // the shift: the median of the medians of three times three elements spread over the row, which a few
      // elements far from the rest (at most one of each three, or all three of one) do not move away from it
      float med[3];
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        const float* p = nf.x + row + (size_t)(3 * u) * ((K - 1) / 8);
        med[u] = __builtin_amdgcn_fmed3f(p[0], p[(K - 1) / 8], p[2 * ((K - 1) / 8)]);
      }
      x0[t] = __builtin_amdgcn_fmed3f(med[0], med[1], med[2]);
    } else {
      x0[t] = 0.f;
    }
    s1[t] = s2[t] = 0.f;
  }
  constexpr int STRIDE = WAVES * 128;
  const int k_full = K & ~127;          // whole steps end here
  const int k_last = k_full - 128;      // the last whole step (negative if there is none)
  if (k_full > 0) {
    // Software pipeline over this wave's steps kb0, kb0 + STRIDE, ...: the weight is fetched two steps
    // ahead and `x` one step ahead; the scheduling barriers keep the fetches of later steps in front of
    // the products of the current one, so a product waits only for its own operands.
    const int kb0 = wave * 128;
    bf16x8 wf[3][RT][4], xf[2][MT][4];
    auto fetch_w = [&](int slot, int kc) {
      const int k = min(kc, k_last);
#pragma unroll
      for (int j = 0; j < RT; ++j)
#pragma unroll
        for (int s = 0; s < 4; ++s) wf[slot][j][s] = load_once(wrow[j] + (size_t)k * W_STEP + W_LOAD * s);
    };
    // NORMED: the float32 elements wait in registers as they came and are shifted, summed and rounded when
    // their step is multiplied, a step after they were asked for (used at once they would make the wave
    // wait for every load before them, the weights' among them)
    f32x4 xr[NORMED ? 2 : 1][MT][4][2];
    auto fetch_x = [&](int slot, int kc) {
      const int k = min(kc, k_last);
      if constexpr (NORM == NORM_OPERAND) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
          xf[slot][0][s] = *(const bf16x8*)((const bf16_t*)normed_rows + min(r, M - 1) * norm_pitch + 8 * g + k + 32 * s);
        return;
      }
      if (NORMED) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            xr[slot][t][s][0] = *(const f32x4*)(xfrow[t] + k + 32 * s);
            xr[slot][t][s][1] = *(const f32x4*)(xfrow[t] + k + 32 * s + 4);
          }
        }
        return;
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) {
#pragma unroll
        for (int s = 0; s < 4; ++s) xf[slot][t][s] = *(const bf16x8*)(xrow[t] + k + 32 * s);
      }
    };
    auto round_x = [&](int slot) {
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          bf16x8 b;
          float a1 = 0.f, a2 = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float v = xr[slot][t][s][e >> 2][e & 3] - x0[t];
            a1 += v;
            a2 = fmaf(v, v, a2);
            b[e] = (bf16_t)v;
          }
          xf[slot][t][s] = b;
          s1[t] += a1;
          s2[t] += a2;
        }
    };
    auto product = [&](int wslot, int xslot) {
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int j = 0; j < RT; ++j)
            acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[wslot][j][s], xf[xslot][t][s], acc[t][j], 0, 0, 0);
    };
    if constexpr (NORM != NORM_OPERAND) fetch_x(0, kb0);
    fetch_w(0, kb0);
    fetch_w(1, kb0 + STRIDE);
    if constexpr (NORM != NORM_NONE) {
      __builtin_amdgcn_sched_barrier(0);
      normed.finish(norm, M, NORM == NORM_OPERAND ? K : N, (bf16_t*)normed_rows, norm_pitch, norm_stat);
      if constexpr (NORM == NORM_OPERAND) {
        __syncthreads();
        fetch_x(0, kb0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // six steps a round, so that every buffer index is a constant (3 weight buffers, 2 x buffers)
    for (int kb = kb0; kb < k_full; kb += 6 * STRIDE) {
#pragma unroll
      for (int u = 0; u < 6; ++u) {
        const int kc = kb + u * STRIDE;
        if (kc < k_full) {
          fetch_x((u + 1) & 1, kc + STRIDE);
          fetch_w((u + 2) % 3, kc + 2 * STRIDE);
          __builtin_amdgcn_sched_barrier(0);
          if (NORMED) round_x(u & 1);
          product(u % 3, u & 1);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
  if (wave == 0 && k_full < K) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = k_full + 32 * s + 8 * g;
      const bool ok = k + 8 <= K;
#pragma unroll
      for (int j = 0; j < RT; ++j) {
        const bf16x8 wv = ok ? *(const bf16x8*)(wrow[j] + (size_t)k_full * W_STEP + W_LOAD * s) : zero;
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          const bf16x8 xv = ok ? *(const bf16x8*)(xrow[t] + k_full + 32 * s) : zero;
          acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xv, acc[t][j], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int j = 0; j < RT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave][t][j][i][lane] = acc[t][j][i];
  if (NORMED) {
    // a row's elements lie with the four lanes that share lane % 16, of every wave
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const float a1 = rows_sum(s1[t]), a2 = rows_sum(s2[t]);
      if (g == 0) {
        stat[wave][t][0][r] = a1;
        stat[wave][t][1][r] = a2;
      }
    }
  }
  __syncthreads();
  if constexpr (GATED) {
    with_gate(act, limit, [&](auto gate) {
      for (int idx = tid; idx < MT * 256; idx += WAVES * 64) {
        const int l = idx & 63, i = (idx >> 6) & 3, t = idx >> 8, m = t * 16 + (l & 15);
        float two[2] = {0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int wv = 0; wv < WAVES; ++wv) two[j] += red[wv][t][j][i][l];
        if (m < M) ((bf16_t*)out)[(size_t)m * (N / 2) + 16 * blockIdx.x + 4 * (l >> 4) + i] = (bf16_t)gate(two[0], two[1]);
      }
    });
    return;
  }
  // acc[t][j][i] of lane l is output column n0 + 16*j + 4*(l/16) + i, row 16*t + l%16.
  auto finish = [&](int idx, int q) {
    const int l = idx & 63, i = (idx >> 6) & 3, j = (idx >> 8) % RT, t = idx / (256 * RT);
    float v = 0.f;
#pragma unroll
    for (int wv = 0; wv < WAVES; ++wv) v += red[wv][t][j][i][l];
    const int n = n0 + 16 * j + 4 * (l >> 4) + i, m = t * 16 + (l & 15);
    // where the scatter turns pairs, the element beside this one (column n ^ 1: the same lane's, i ^ 1) as well
    const bool pairs = QKV && sc.turn_a != nullptr;
    float beside = 0.f;
    if (pairs) {
#pragma unroll
      for (int wv = 0; wv < WAVES; ++wv) beside += red[wv][t][j][i ^ 1][l];
    }
    if (NORMED && n < N) {
      float a1 = 0.f, a2 = 0.f;
#pragma unroll
      for (int wv = 0; wv < WAVES; ++wv) {
        a1 += stat[wv][t][0][l & 15];
        a2 += stat[wv][t][1][l & 15];
      }
      const float mean = nf.center ? a1 / (float)K : 0.f;     // of x - x0
      const float var = fmaxf(a2 / (float)K - mean * mean, 0.f);
      const float rstd = rsqrtf(var + nf.eps);
      v = rstd * (v - mean * (EARLY ? fold_c[q] : nf.c[n])) + (EARLY ? fold_d[q] : nf.d[n]);
      if (pairs) beside = rstd * (beside - mean * nf.c[n ^ 1]) + nf.d[n ^ 1];
    }
    if (n < N && m < M) {
      if (QKV) {
        if (bias) {
          v += EARLY ? add[q] : bias[n];
          if (pairs) beside += bias[n ^ 1];
        }
        qkv_store(v, beside, m, n, sc, EARLY ? page[q] : sc.token_page[m], EARLY ? off[q] : sc.token_off[m]);
      } else if (EARLY) {
        if (bias) v += add[q];
        v = apply_act(v, act);
        if (NORM == NORM_RESIDUAL) v += (onto[q] - norm_stat[m][0]) * norm_stat[m][1] * onto_w[q] + onto_b[q];
        else if constexpr (PAIRS) {
          float o = onto[q];
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (c < top) o += of_pair[q][c];
          v += o;
        } else if (residual) v += onto[q];
        store_any(out, out_dtype, (size_t)m * N + n, v);
      } else {
        epilogue_store(v, m, n, N, bias, residual, out, out_dtype, act);
      }
    }
  };
  if constexpr (EARLY) {
#pragma unroll
    for (int q = 0; q < OUTS; ++q) finish(tid + q * WAVES * 64, q);
  } else {
    for (int idx = tid; idx < MT * RT * 256; idx += WAVES * 64) finish(idx, 0);
  }
}

template <int MT, int WAVES, int RT>
static void launch_skinny(const bf16_t* xp, const bf16_t* wp, const bf16_t* ws, const float* bias,
                          const float* residual, void* out, int out_dtype, int act, int M, int N, int K,
                          const QkvScatter* sc, const NormFold* nf, hipStream_t stream) {
  const dim3 grid((N + 16 * RT - 1) / (16 * RT)), block(WAVES * 64);
  const QkvScatter none{};
  const NormFold plain{};
  if (nf) {           // the dispatcher has seen to it that there is a tile-ordered weight and MT <= 2
    if constexpr (MT <= 2) {
      if (sc)
        gemm_bf16_skinny_kernel<MT, WAVES, true, true, RT, true><<<grid, block, 0, stream>>>(
            nullptr, ws, bias, residual, out, out_dtype, act, M, N, K, *sc, *nf, NoNorm{});
      else
        gemm_bf16_skinny_kernel<MT, WAVES, false, true, RT, true><<<grid, block, 0, stream>>>(
            nullptr, ws, bias, residual, out, out_dtype, act, M, N, K, none, *nf, NoNorm{});
    }
    return;
  }
  if (ws && sc)
    gemm_bf16_skinny_kernel<MT, WAVES, true, true, RT><<<grid, block, 0, stream>>>(xp, ws, bias, residual, out,
                                                                                out_dtype, act, M, N, K, *sc, plain, NoNorm{});
  else if (ws)
    gemm_bf16_skinny_kernel<MT, WAVES, false, true, RT><<<grid, block, 0, stream>>>(xp, ws, bias, residual, out,
                                                                                 out_dtype, act, M, N, K, none, plain, NoNorm{});
  else if (sc)
    gemm_bf16_skinny_kernel<MT, WAVES, true, false, RT><<<grid, block, 0, stream>>>(xp, wp, bias, residual, out,
                                                                                 out_dtype, act, M, N, K, *sc, plain, NoNorm{});
  else
    gemm_bf16_skinny_kernel<MT, WAVES, false, false, RT><<<grid, block, 0, stream>>>(xp, wp, bias, residual, out,
                                                                                  out_dtype, act, M, N, K, none, plain, NoNorm{});
}

// The same next to a norm (see `RowNorm`), up to 8 rows, from the tile-ordered weight.
template <int RT, int NORM, int ROWS, int PER>
static void launch_skinny_norm(const bf16_t* xp, const bf16_t* ws, const float* bias, void* out, int out_dtype, int act, int M, int N,
                               int K, const QkvScatter* sc, const RowNorm& norm, hipStream_t stream) {
  const dim3 grid((N + 16 * RT - 1) / (16 * RT));
  const unsigned lds = NORM == NORM_OPERAND ? M * (K + 8) * 2 : 0;
  // (8 rows of 3,072 and what the kernel has beside them are 62 KB: no more than any launch may ask for)
  if constexpr (NORM == NORM_OPERAND) {
    if (sc) {
      gemm_bf16_skinny_kernel<1, 4, true, true, RT, false, NORM, ROWS, PER><<<grid, 256, lds, stream>>>(
          nullptr, ws, bias, nullptr, out, out_dtype, act, M, N, K, *sc, NormFold{}, norm);
      return;
    }
  }
  gemm_bf16_skinny_kernel<1, 4, false, true, RT, false, NORM, ROWS, PER><<<grid, 256, lds, stream>>>(
      xp, ws, bias, nullptr, out, out_dtype, act, M, N, K, QkvScatter{}, NormFold{}, norm);
}
template <int RT, int NORM>
static void skinny_norm_rows(const bf16_t* xp, const bf16_t* ws, const float* bias, void* out, int out_dtype, int act, int M, int N, int K,
                            const QkvScatter* sc, const RowNorm& norm, hipStream_t stream) {
  const int width = NORM == NORM_OPERAND ? K : N;       // (registers for the rows as they are)
#define SKINNY_NORM(PER)                                                                                                             \
  if (M <= 4) launch_skinny_norm<RT, NORM, 1, PER>(xp, ws, bias, out, out_dtype, act, M, N, K, sc, norm, stream);                  \
  else launch_skinny_norm<RT, NORM, 2, PER>(xp, ws, bias, out, out_dtype, act, M, N, K, sc, norm, stream)
  if (width <= 1024) { SKINNY_NORM(4); return; }
  if constexpr (NORM == NORM_OPERAND)
    if (width > 2048) { SKINNY_NORM(12); return; }
  SKINNY_NORM(8);
#undef SKINNY_NORM
}
template <int RT>
static void skinny_norm(int kind, const bf16_t* xp, const bf16_t* ws, const float* bias, void* out, int out_dtype, int act, int M, int N,
                       int K, const QkvScatter* sc, const RowNorm& norm, hipStream_t stream) {
  if (kind == NORM_OPERAND) skinny_norm_rows<RT, NORM_OPERAND>(xp, ws, bias, out, out_dtype, act, M, N, K, sc, norm, stream);
  else skinny_norm_rows<RT, NORM_RESIDUAL>(xp, ws, bias, out, out_dtype, act, M, N, K, sc, norm, stream);
}

// How many tiles of 16 weight rows a block of the few-rows kernel takes (1, 2 or 3). Every block reads all of
// `x`, so fewer and larger blocks read less of it; what decides is how evenly the blocks fall on the compute
// units, which take them in turns: the launch takes what the fullest unit gets, ceil(blocks / units) blocks of
// `tiles` tiles and one reading of `x` each, which costs about a fortieth of a tile for every row of `x`
// (lanes beyond the last row read it again, from the cache), and among equals the larger blocks win.
// 12,288 columns on 256 units: 768, 384 or 256 blocks, 3, 4 or 3 tiles a unit: 21.2 us with one tile a block,
// 20.5 with three; 9,216 columns and K = 36,864: 576, 288 or 192 blocks, again 3, 4 or 3: 139, 159 and 114 us;
// 20,480 columns, K = 5,120: 5, 6 and 6 tiles a unit, and one tile a block is quickest at 8 rows (39.6 us
// against 41.3 with three), three tiles at 16 rows (45.7 against 48.9 with one). With blocks for four rounds or
// more the units even out by themselves. Three tiles up to 16 rows of `x`, two up to 32.
static int skinny_tiles_per_block(int M, int N) {
  if (M > 32) return 1;
  const int units = tnx_compute_units();
  const int tiles = (N + 15) / 16;
  const float x_cost = 0.025f * (float)min(M, 16);
  int best = 1;
  float best_cost = (float)((tiles + units - 1) / units) * (1.f + x_cost);
  for (int rt = 2; rt <= (M <= 16 ? 3 : 2); ++rt) {
    const int blocks = (tiles + rt - 1) / rt;
    if (blocks >= 4 * units) {
      best = rt;
      continue;
    }
    const float cost = (float)((blocks + units - 1) / units) * ((float)rt + x_cost);
    if (2 * blocks >= units && cost <= best_cost + 1e-3f) {
      best = rt;
      best_cost = cost;
    }
  }
  return best;
}

extern "C" int tnx_gemm_skinny_tiles_per_block(int M, int N) { return skinny_tiles_per_block(M, N); }

static int gemm_bf16_dispatch(const void* x, const void* w, const void* w_tiles, const float* bias,
                              const float* residual, void* out, int out_dtype, int act, int M, int N, int K,
                              int force_tiled, const QkvScatter* sc, hipStream_t stream,
                              const NormFold* nf = nullptr) {
  TNX_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_bf16: bad sizes M=%d N=%d K=%d", M, N, K);
  if (nf) {
    TNX_REQUIRE(w_tiles != nullptr && M <= 32 && K % 128 == 0 && N % 16 == 0 && force_tiled != 1,
                "gemm_bf16: a product of normalised rows takes up to 32 rows and a tile-ordered weight, K a "
                "multiple of 128 and N of 16; got M=%d N=%d K=%d", M, N, K);
    TNX_REQUIRE(((uintptr_t)nf->x | (uintptr_t)w_tiles) % 16 == 0, "gemm_bf16: operands must be 16-byte aligned");
    x = w = w_tiles;          // what the checks below look at
  }
  TNX_REQUIRE(K % 8 == 0, "gemm_bf16: the inner size K=%d must be a multiple of 8", K);
  TNX_REQUIRE(((uintptr_t)x | (uintptr_t)w) % 16 == 0, "gemm_bf16: operands must be 16-byte aligned");
  if (M == 0) return 0;
  const bf16_t* xp = (const bf16_t*)x;
  const bf16_t* wp = (const bf16_t*)w;
  const bf16_t* ws = (const bf16_t*)w_tiles;
  TNX_REQUIRE(ws == nullptr || (N % 16 == 0 && K % 128 == 0),
              "gemm_bf16: a tile-ordered weight needs N a multiple of 16 and K of 128, got N=%d K=%d", N, K);
  // The few-rows kernel up to 32 rows (beyond that every block reading all of `x` again costs more than the
  // tiles' detour through LDS: 245 against 151 us for the 50,272 x 4,096 head at 64 rows), or when asked for.
  if ((M <= 32 || ((force_tiled == 4 || force_tiled == 8) && M <= 64)) && force_tiled != 1) {
    // Four waves a block (eight, for the few blocks of a narrow matrix with a long K, are no quicker anywhere
    // and 5 to 8 % slower at 2,048 x 8,192 to 3,072 x 12,288). force_tiled 4 or 8 picks the wave count and 2
    // or 3 the tiles a block, for measurements and tests.
    const int waves = force_tiled == 8 ? 8 : 4;
    const int tiles_per_block = force_tiled == 0 && waves == 4 ? skinny_tiles_per_block(M, N) : 1;
    const bool two_tiles = force_tiled == 2 || tiles_per_block == 2;
    const bool three_tiles = tiles_per_block == 3;
#define SKINNY(MT, WV, RT) \
  launch_skinny<MT, WV, RT>(xp, wp, ws, bias, residual, out, out_dtype, act, M, N, K, sc, nf, stream)
#define SKINNY_MT(WV)                        \
  switch ((M + 15) / 16) {                   \
    case 1: SKINNY(1, WV, 1); break;         \
    case 2: SKINNY(2, WV, 1); break;         \
    case 3: SKINNY(3, WV, 1); break;         \
    default: SKINNY(4, WV, 1); break;        \
  }
    if ((force_tiled == 3 || three_tiles) && M <= 16) {
      SKINNY(1, 4, 3);
    } else if (force_tiled == 5 && M <= 16) {
      SKINNY(1, 8, 2);
    } else if (force_tiled == 6 && M <= 16) {
      SKINNY(1, 8, 3);
    } else if (two_tiles && M <= 16) {
      SKINNY(1, 4, 2);
    } else if (two_tiles && M <= 32) {
      SKINNY(2, 4, 2);
    } else if (waves == 8) {
      SKINNY_MT(8);
    } else {
      SKINNY_MT(4);
    }
#undef SKINNY_MT
#undef SKINNY
    TNX_CHECK_LAUNCH("gemm_bf16_skinny");
    return 0;
  }
  if (!sc && force_tiled != 1 && wide_tiles_fit(M, N, K, residual, out_dtype, act) && (uintptr_t)out % 16 == 0 &&
      (uintptr_t)residual % 16 == 0 && (uintptr_t)bias % 16 == 0) {
    const int rc = launch_wide(xp, wp, bias, residual, out, out_dtype, act, M, N, K, stream);
    if (rc) return rc;
    TNX_CHECK_LAUNCH("gemm_bf16_wide");
    return 0;
  }
  dim3 grid((N + BT_N - 1) / BT_N, (M + BT_M - 1) / BT_M);
  TNX_REQUIRE(grid.y <= 65535, "gemm_bf16: M=%d is too large", M);
  if (sc)
    gemm_bf16_kernel<true><<<grid, 256, 0, stream>>>(xp, wp, bias, residual, out, out_dtype, act, M, N, K, *sc);
  else
    gemm_bf16_kernel<false><<<grid, 256, 0, stream>>>(xp, wp, bias, residual, out, out_dtype, act, M, N, K,
                                                      QkvScatter{});
  TNX_CHECK_LAUNCH("gemm_bf16");
  return 0;
}

// x w^T + residual + each row's `top` rows of `pairs` [M top, N], float32, up to 16 rows, from the tile-ordered copy.
extern "C" int tnx_gemm_bf16_pairs(const void* x, const void* w_tiles, const float* residual, const float* pairs, int top, float* out, int M,
                                   int N, int K, hipStream_t stream) {
  TNX_REQUIRE(M >= 0 && M <= 16 && N > 0 && N % 16 == 0 && K > 0 && K % 128 == 0 && top >= 1 && top <= 4,
              "gemm_bf16_pairs: up to 16 rows of up to 4 pairs, N in 16s, K in 128s, got M=%d N=%d K=%d, %d", M, N, K, top);
  TNX_REQUIRE(((uintptr_t)x | (uintptr_t)w_tiles) % 16 == 0, "gemm_bf16_pairs: operands must be 16-byte aligned");
  if (M == 0) return 0;
#define PAIRS_SKINNY(RT)                                                                                                               \
  gemm_bf16_skinny_kernel<1, 4, false, true, RT, false, NORM_NONE, 1, 1, false, true><<<dim3((N / 16 + RT - 1) / RT), 256, 0, stream>>>( \
      (const bf16_t*)x, (const bf16_t*)w_tiles, nullptr, residual, out, TNX_F32, TNX_ACT_NONE, M, N, K, QkvScatter{}, NormFold{},        \
      NoNorm{}, 0.f, pairs, top)
  switch (skinny_tiles_per_block(M, N)) {
    case 1: PAIRS_SKINNY(1); break;
    case 2: PAIRS_SKINNY(2); break;
    default: PAIRS_SKINNY(3); break;
  }
#undef PAIRS_SKINNY
  TNX_CHECK_LAUNCH("gemm_bf16_pairs");
  return 0;
}

// act(g) * u of the product with gate rows and as many up rows (N together), up to 32 rows, from the tile-ordered copy; bfloat16.
extern "C" int tnx_gated_activation_skinny(const void* x, const void* w_tiles, void* out, int act, float limit, int M, int N, int K,
                                           hipStream_t stream) {
  TNX_REQUIRE(M >= 0 && M <= 32 && N > 0 && N % 32 == 0 && K > 0 && K % 128 == 0,
              "gated_activation_skinny: up to 32 rows, N in 32s, K in 128s, got M=%d N=%d K=%d", M, N, K);
  TNX_REQUIRE(((uintptr_t)x | (uintptr_t)w_tiles) % 16 == 0, "gated_activation_skinny: operands must be 16-byte aligned");
  if (M == 0) return 0;
#define GATED_SKINNY(MT)                                                                                                     \
  gemm_bf16_skinny_kernel<MT, 4, false, true, 2, false, NORM_NONE, 1, 1, true><<<dim3(N / 32), 256, 0, stream>>>(            \
      (const bf16_t*)x, (const bf16_t*)w_tiles, nullptr, nullptr, out, TNX_BF16, act, M, N, K, QkvScatter{}, NormFold{}, NoNorm{}, limit)
  if (M <= 16) GATED_SKINNY(1);
  else GATED_SKINNY(2);
#undef GATED_SKINNY
  TNX_CHECK_LAUNCH("gated_activation_skinny");
  return 0;
}

// `w_tiles` (optional) is the tile-ordered copy of `w` that the few-rows kernel streams faster.
extern "C" int tnx_gemm_bf16(const void* x, const void* w, const void* w_tiles, const float* bias,
                             const float* residual, void* out, int out_dtype, int act, int M, int N, int K,
                             int force_tiled, hipStream_t stream) {
  return gemm_bf16_dispatch(x, w, w_tiles, bias, residual, out, out_dtype, act, M, N, K, force_tiled, nullptr,
                            stream);
}

// The fused projection of queries, keys and values: `x w^T + bias` with w = [Wq; Wk; Wv] stacked by rows,
// queries scaled and written densely, keys and values written straight into their cache pages.
// What both forms of the fused projection check and fill in of the pair-turning tables.
template <typename T>
static int qkv_turn(QkvScatterOf<T>& sc, const float* turn_a, const float* turn_b, const int* positions, int turn_rows,
                    int page_pad) {
  TNX_REQUIRE(page_pad >= 0 && page_pad % 8 == 0, "gemm_bf16_qkv: bad distance between pages");
  sc.page_pad = page_pad;
  TNX_REQUIRE((turn_a == nullptr) == (turn_b == nullptr), "gemm_bf16_qkv: the pair-turning tables come both or not at all");
  TNX_REQUIRE(!turn_a || (positions && turn_rows > 0 && sc.head_size % 2 == 0),
              "gemm_bf16_qkv: pair-turning tables need the tokens' positions, rows, and an even head size");
  sc.turn_a = turn_a;
  sc.turn_b = turn_b;
  sc.positions = positions;
  sc.turn_rows = turn_rows;
  return 0;
}

extern "C" int tnx_gemm_bf16_qkv(const void* x, const void* w, const void* w_tiles, const float* bias, int M, int K,
                                 const int* token_page,
                                 const int* token_off, void* q_out, void* k_pages, void* v_pages, float scale,
                                 int num_heads, int num_kv, int head_size, int page_size, int num_pages,
                                 int force_tiled, const float* turn_a, const float* turn_b, const int* positions,
                                 int turn_rows, int page_pad, hipStream_t stream) {
  TNX_REQUIRE(num_heads > 0 && num_kv >= 0 && head_size > 0 && page_size > 0, "gemm_bf16_qkv: bad sizes");
  QkvScatter sc;
  sc.token_page = token_page;
  sc.token_off = token_off;
  sc.q_out = (bf16_t*)q_out;
  sc.k_pages = (bf16_t*)k_pages;
  sc.v_pages = (bf16_t*)v_pages;
  sc.scale = scale;
  sc.nq = num_heads * head_size;
  sc.nk = num_kv * head_size;
  sc.head_size = head_size;
  sc.num_kv = num_kv;
  sc.page_size = page_size;
  sc.num_pages = num_pages;
  if (int rc = qkv_turn(sc, turn_a, turn_b, positions, turn_rows, page_pad)) return rc;
  const int N = sc.nq + 2 * sc.nk;
  return gemm_bf16_dispatch(x, w, w_tiles, bias, nullptr, nullptr, TNX_BF16, TNX_ACT_NONE, M, N, K, force_tiled, &sc,
                            stream);
}

// The float32 engine's, for up to 16 rows and K of a multiple of 4.
extern "C" int tnx_gemm_f32_qkv(const float* x, const float* w, const float* bias, int M, int K, const int* token_page,
                                const int* token_off, float* q_out, float* k_pages, float* v_pages, float scale,
                                int num_heads, int num_kv, int head_size, int page_size, int num_pages,
                                const float* turn_a, const float* turn_b, const int* positions, int turn_rows, int page_pad,
                                hipStream_t stream) {
  TNX_REQUIRE(num_heads > 0 && num_kv >= 0 && head_size > 0 && head_size % 4 == 0 && page_size > 0, "gemm_f32_qkv: bad sizes");
  TNX_REQUIRE(M >= 0 && M <= 16 && K > 0 && K % 4 == 0 && ((uintptr_t)x | (uintptr_t)w) % 16 == 0,
              "gemm_f32_qkv: up to 16 rows that begin at multiples of 16 bytes, got %d of %d", M, K);
  QkvScatterOf<float> sc{token_page, token_off, q_out, k_pages, v_pages, scale, num_heads * head_size, num_kv * head_size,
                         head_size, num_kv, page_size, num_pages};
  if (int rc = qkv_turn(sc, turn_a, turn_b, positions, turn_rows, page_pad)) return rc;
  if (M == 0) return 0;
  f32_skinny(x, w, bias, nullptr, nullptr, TNX_F32, TNX_ACT_NONE, M, sc.nq + 2 * sc.nk, K, sc, stream);
  TNX_CHECK_LAUNCH("gemm_f32_qkv");
  return 0;
}

// Products of up to 8 rows next to a norm (see `RowNorm`), `w` in tile order. `kind` NORM_OPERAND: x is what `norm` gives (its
// width is K); NORM_RESIDUAL: what it gives is added to the result (its width is N).
static int norm_fits(int kind, const RowNorm* norm, const void* w, int M, int N, int K) {
  TNX_REQUIRE(norm && norm->x && (kind == NORM_OPERAND || kind == NORM_RESIDUAL), "product next to a norm: no norm");
  const int width = kind == NORM_OPERAND ? K : N, most = kind == NORM_OPERAND ? NORM_OPERAND_WIDTH : NORM_RESIDUAL_WIDTH;
  TNX_REQUIRE(width <= most && norm->eps > 0.f &&
              ((uintptr_t)norm->x | (uintptr_t)norm->weight | (uintptr_t)norm->bias | (uintptr_t)w) % 16 == 0,
              "product next to a norm: rows of up to %d that begin at multiples of 16 bytes, got %d", most, width);
  TNX_REQUIRE(M > 0 && M <= 8 && N > 0 && N % 16 == 0 && K > 0 && K % 128 == 0, "product next to a norm: bad sizes M=%d N=%d K=%d", M, N, K);
  return 0;
}

extern "C" int tnx_gemm_bf16_by_norm(int kind, const RowNorm* norm, const void* x, const void* w, const float* bias, void* out,
                                     int out_dtype, int act, int M, int N, int K, hipStream_t stream) {
  if (int rc = norm_fits(kind, norm, w, M, N, K)) return rc;
  TNX_REQUIRE(kind == NORM_OPERAND || (x && (uintptr_t)x % 16 == 0), "product next to a norm: its rows begin at multiples of 16 bytes");
  const bf16_t *xp = (const bf16_t*)x, *ws = (const bf16_t*)w;
  const int tiles = skinny_tiles_per_block(M, N);
#define BY_NORM(RT) skinny_norm<RT>(kind, xp, ws, bias, out, out_dtype, act, M, N, K, nullptr, *norm, stream)
  if (tiles == 3) BY_NORM(3); else if (tiles == 2) BY_NORM(2); else BY_NORM(1);
#undef BY_NORM
  TNX_CHECK_LAUNCH("gemm_bf16_by_norm");
  return 0;
}

// Queries, keys and values of what a norm gives, straight to their places.
extern "C" int tnx_gemm_bf16_by_norm_qkv(const RowNorm* norm, const void* w, const float* bias, int M, int K, const int* token_page,
                                         const int* token_off, void* q_out, void* k_pages, void* v_pages, float scale, int num_heads,
                                         int num_kv, int head_size, int page_size, int num_pages, const float* turn_a,
                                         const float* turn_b, const int* positions, int turn_rows, int page_pad, hipStream_t stream) {
  TNX_REQUIRE(num_heads > 0 && num_kv >= 0 && head_size > 0 && page_size > 0, "gemm_bf16_by_norm_qkv: bad sizes");
  const int nq = num_heads * head_size, nk = num_kv * head_size, N = nq + 2 * nk;
  if (int rc = norm_fits(NORM_OPERAND, norm, w, M, N, K)) return rc;
  QkvScatter sc{token_page, token_off, (bf16_t*)q_out, (bf16_t*)k_pages, (bf16_t*)v_pages, scale, nq, nk, head_size, num_kv, page_size, num_pages};
  if (int rc = qkv_turn(sc, turn_a, turn_b, positions, turn_rows, page_pad)) return rc;
  const bf16_t* ws = (const bf16_t*)w;
  const int tiles = skinny_tiles_per_block(M, N);
#define BY_NORM(RT) skinny_norm<RT>(NORM_OPERAND, nullptr, ws, bias, nullptr, TNX_BF16, TNX_ACT_NONE, M, N, K, &sc, *norm, stream)
  if (tiles == 3) BY_NORM(3); else if (tiles == 2) BY_NORM(2); else BY_NORM(1);
#undef BY_NORM
  TNX_CHECK_LAUNCH("gemm_bf16_by_norm_qkv");
  return 0;
}

// The same two for the rows of a LayerNorm's input (float32), the norm folded into the product (see `NormFold`):
// `w_folded` is W diag(gamma) in tile order, `fold_c` its row sums, `fold_d` W beta.
extern "C" int tnx_gemm_bf16_normed(const float* x, const void* w_folded, const float* fold_c, const float* fold_d,
                                    float eps, const float* bias, void* out, int out_dtype, int act, int M, int N,
                                    int K, int force_tiled, int center, hipStream_t stream) {
  const NormFold nf{x, fold_c, fold_d, eps, center};
  return gemm_bf16_dispatch(nullptr, nullptr, w_folded, bias, nullptr, out, out_dtype, act, M, N, K, force_tiled,
                            nullptr, stream, &nf);
}

extern "C" int tnx_gemm_bf16_qkv_normed(const float* x, const void* w_folded, const float* fold_c,
                                        const float* fold_d, float eps, const float* bias, int M, int K,
                                        const int* token_page, const int* token_off, void* q_out, void* k_pages,
                                        void* v_pages, float scale, int num_heads, int num_kv, int head_size,
                                        int page_size, int num_pages, int force_tiled, const float* turn_a,
                                        const float* turn_b, const int* positions, int turn_rows, int page_pad,
                                        int center, hipStream_t stream) {
  TNX_REQUIRE(num_heads > 0 && num_kv >= 0 && head_size > 0 && page_size > 0, "gemm_bf16_qkv: bad sizes");
  QkvScatter sc;
  sc.token_page = token_page;
  sc.token_off = token_off;
  sc.q_out = (bf16_t*)q_out;
  sc.k_pages = (bf16_t*)k_pages;
  sc.v_pages = (bf16_t*)v_pages;
  sc.scale = scale;
  sc.nq = num_heads * head_size;
  sc.nk = num_kv * head_size;
  sc.head_size = head_size;
  sc.num_kv = num_kv;
  sc.page_size = page_size;
  sc.num_pages = num_pages;
  if (int rc = qkv_turn(sc, turn_a, turn_b, positions, turn_rows, page_pad)) return rc;
  const int N = sc.nq + 2 * sc.nk;
  const NormFold nf{x, fold_c, fold_d, eps, center};
  return gemm_bf16_dispatch(nullptr, nullptr, w_folded, bias, nullptr, nullptr, TNX_BF16, TNX_ACT_NONE, M, N, K,
                            force_tiled, &sc, stream, &nf);
}

// ------------------------------------------------------------------------------------------ bfloat16, some rows
//
// Decode batches beyond the few-rows kernel (33 to 128 rows): the product is still the weight read once, but
// every block of the few-rows kernel would read all of `x` again, and the vendor library's kernels for such
// sizes leave much of the memory's rate unused where the output is small and K long (the products that end
// in the residual sum). Here a block of four waves takes 64 weight rows (each wave a tile of 16, from the
// tile-ordered copy in runs of 1 KB) and one share of K. Everything comes straight from global memory into
// LDS, AHEAD steps of 128 before it is used: the rows of `x` once a block, 16-byte chunks swizzled over the
// 256 bytes of a row, and each wave's weights into a place of its own, where a lane finds the 16 bytes it
// asked for (row lane % 16, chunk lane / 16 of the tile's step). No load lands in a register, so the only waits are the ones written here, and AHEAD - 1 whole
// steps stay in flight while one is multiplied. The shares of K (gridDim.y of them, so that the blocks fill
// the chip also where N is small) leave their float32 partial sums in a workspace [shares][M][N] that a
// second kernel adds up in a fixed order, with bias, activation and residual; one share alone writes the
// result itself.
template <int MT, int AHEAD, int NW, typename Scatter>
__global__ void __launch_bounds__(64 * NW)
gemm_bf16_mid_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w_tiles, const float* __restrict__ bias,
                     const float* __restrict__ residual, void* __restrict__ out, int out_dtype, int act,
                     float* __restrict__ partial, int M, int N, int K, int steps_per_share, Scatter sc) {
  constexpr bool SCATTER = !std::is_same<Scatter, NoScatter>::value;
  extern __shared__ __attribute__((aligned(16))) char mid_smem[];
  constexpr int NST = AHEAD + 1;                    // stages: the step that is multiplied and those in flight
  constexpr int XSTAGE = 16 * MT * 256;             // bytes of a step's rows of x
  constexpr int WSTAGE = 4 * 1024;                  // bytes of a step's weights of one wave
  constexpr int XLOADS = (4 * MT + NW - 1) / NW;    // loads of x of a wave a step (where they do not come out even, some twice)
  constexpr int LOADS = XLOADS + 4;                 // loads of a wave a step
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int share = blockIdx.y;
  const int steps_all = K / 128;
  const int step0 = share * steps_per_share;
  const int steps = min(steps_per_share, steps_all - step0);      // at least one: the host cuts no empty share
  const int last = step0 + steps - 1;
  const int tile = blockIdx.x * NW + wave;          // this wave's tile of 16 weight rows
  const char* wtile = (const char*)(w_tiles + (size_t)min(tile, N / 16 - 1) * 16 * K);
  // the loads of x: wave-load u of this wave brings rows 4 q .. 4 q + 3 (q = wave + NW u), 16 lanes a row; the
  // lane at place p of row m brings chunk p ^ (m % 16), so that fragment reads meet no bank twice
  unsigned xoff[XLOADS];
#pragma unroll
  for (int u = 0; u < XLOADS; ++u) {
    const int row = 4 * min(wave + NW * u, 4 * MT - 1) + (lane >> 4);
    xoff[u] = (unsigned)(((size_t)min(row, M - 1) * K + (((lane & 15) ^ (row & 15)) * 8)) * 2);
  }
  const unsigned x_lds = lds_offset(mid_smem);
  const unsigned w_lds = x_lds + NST * XSTAGE + wave * NST * WSTAGE;
  const char* w_mine = mid_smem + NST * XSTAGE + wave * NST * WSTAGE;
  auto issue = [&](int stage, int step) {
    const int st = min(step, last);                 // beyond the share: the last step again, into a stage nobody reads
    const char* xbase = (const char*)(x + (size_t)st * 128);
#pragma unroll
    for (int u = 0; u < XLOADS; ++u)
      load_to_lds(xbase, xoff[u], x_lds + stage * XSTAGE + min(wave + NW * u, 4 * MT - 1) * 1024);
    const char* wbase = wtile + (size_t)st * (128 * 16 * 2);
#pragma unroll
    for (int s = 0; s < 4; ++s) load_to_lds_once(wbase + 1024 * s, (unsigned)((r * 4 + g) * 16), w_lds + stage * WSTAGE + 1024 * s);
  };
  // What the end adds, and where its results go, asked for before the products, and results stored four at a time: behind the
  // products they were another time to memory, and sixteen stores of 2 bytes a row. Steps of 2.7b with 32 requests of 700 tokens
  // 3,437 / 3,298 us, before and after.
  const int n = 16 * tile + 4 * g, shares = gridDim.y;
  f32x4 add = {0.f, 0.f, 0.f, 0.f};
  int page[SCATTER ? MT : 1], off[SCATTER ? MT : 1];
  if (bias && shares == 1) {
#pragma unroll
    for (int e = 0; e < 4; ++e) add[e] = bias[min(n + e, N - 1)];
  }
  if constexpr (SCATTER) {
#pragma unroll
    for (int t = 0; t < MT; ++t) page[t] = sc.token_page[min(16 * t + r, M - 1)], off[t] = sc.token_off[min(16 * t + r, M - 1)];
  }
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto products = [&](int stage) {
    const char* xs = mid_smem + stage * XSTAGE;
    const char* ws = w_mine + stage * WSTAGE + lane * 16;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const bf16x8 wf = *(const bf16x8*)(ws + 1024 * s);
      bf16x8 xf[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) xf[t] = *(const bf16x8*)(xs + (16 * t + r) * 256 + (((4 * s + g) ^ r) * 16));
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf[t], acc[t], 0, 0, 0);
    }
  };
#pragma unroll
  for (int a = 0; a < AHEAD; ++a) issue(a, step0 + a);
  for (int i0 = 0; i0 < steps; i0 += NST) {
#pragma unroll
    for (int u = 0; u < NST; ++u) {
      if (i0 + u < steps) {
        // step i has landed when only the loads of the AHEAD - 1 steps after it are in flight
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AHEAD - 1) * LOADS) : "memory");
        __syncthreads();        // its rows of x are there for all; and all have done with the stage of step i - 1,
        issue((u + AHEAD) % NST, step0 + i0 + u + AHEAD);      // where step i + AHEAD goes
        products(u);
      }
    }
  }
  wait_for_loads();             // the loads beyond the last step write to LDS: they end before the block does
  // acc[t][e] of a lane is row m = 16 t + r of the output at column 16 tile + 4 g + e
  if (!SCATTER && shares == 1)
    with_act(act, [&](auto activation) {
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][e] = activation(acc[t][e] + add[e]);
    });
  if (n < N) {
    bool fours = ((uintptr_t)out & 15) == 0;
    if constexpr (SCATTER) fours = qkv_in_fours(sc);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int m = 16 * t + r;
      if (m >= M) continue;
      if constexpr (SCATTER) {
        const f32x4 v = acc[t] + add;
        if (fours) {
          qkv_store_four(v, m, n, sc, page[t], off[t]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) qkv_store(v[e], v[e ^ 1], m, n + e, sc, page[t], off[t]);
        }
      } else if (shares == 1) {
        f32x4 v = acc[t];
        const size_t o = (size_t)m * N + n;
        if (residual) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += residual[o + e];
        }
        store_four(v, out, out_dtype, o, fours);
      } else {
        *(f32x4*)(partial + ((size_t)share * M + m) * N + n) = acc[t];
      }
    }
  }
}

// out = act(sum over the shares + bias) + residual, four columns a thread, the shares in their order.
// (Leaving this sum to the LayerNorm that reads the rows next, in one launch with it, was measured at 64 rows of
// 4,096: this kernel's 4.9 us went, but the norm, a block a row, then pulled 100 KB a block through 64 compute
// units and took 9.1 us in place of 6.0; the step stayed as it was.)
__global__ void __launch_bounds__(256)
gemm_mid_sum_kernel(const float* __restrict__ partial, const float* __restrict__ bias,
                    const float* __restrict__ residual, void* __restrict__ out, int out_dtype, int act, int M, int N,
                    int shares) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= (size_t)M * N) return;
  const int m = (int)(i / N), n = (int)(i - (size_t)m * N);
  // (bias and residual before the shares: behind them they would be waited for once more; N is a multiple of 4)
  const bool fours = (((uintptr_t)bias | (uintptr_t)residual | (uintptr_t)out) & 15) == 0;
  f32x4 add = {0.f, 0.f, 0.f, 0.f}, onto = {0.f, 0.f, 0.f, 0.f};
  if (fours) {
    if (bias) add = *(const f32x4*)(bias + n);
    if (residual) onto = *(const f32x4*)(residual + i);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (bias) add[e] = bias[n + e];
      if (residual) onto[e] = residual[i + e];
    }
  }
  f32x4 v;
  // every share is asked for before the first is added, so that the kernel waits for memory once; the order of the sum stays
  // (up to eight, shares beyond the last read the last one again and are left out)
  if (shares <= 8) {
    f32x4 p[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) p[s] = *(const f32x4*)(partial + (size_t)min(s, shares - 1) * M * N + i);
    v = p[0];
#pragma unroll
    for (int s = 1; s < 8; ++s)
      if (s < shares) v += p[s];
  } else if (shares <= 16) {
    f32x4 p[16];
#pragma unroll
    for (int s = 0; s < 16; ++s)
      if (s < shares) p[s] = *(const f32x4*)(partial + (size_t)s * M * N + i);
    v = p[0];
#pragma unroll
    for (int s = 1; s < 16; ++s)
      if (s < shares) v += p[s];
  } else {
    v = *(const f32x4*)(partial + i);
    for (int s = 1; s < shares; ++s) v += *(const f32x4*)(partial + (size_t)s * M * N + i);
  }
  v += add;
  with_act(act, [&](auto activation) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = activation(v[e]);
  });
  store_four(v + onto, out, out_dtype, i, fours);
}

template <int MT, int AHEAD, int NW = 4, typename Scatter = NoScatter>
static int launch_mid(const bf16_t* x, const bf16_t* w_tiles, const float* bias, const float* residual, void* out,
                      int out_dtype, int act, float* partial, int M, int N, int K, int shares, int* left, hipStream_t stream,
                      const Scatter& sc = Scatter{}) {
  constexpr int bytes = (AHEAD + 1) * (16 * MT * 256 + NW * 4 * 1024);
  static_assert(bytes <= 160 * 1024, "the stages do not fit the LDS of a compute unit");
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_bf16_mid_kernel<MT, AHEAD, NW, Scatter>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) {
      tnx_set_error("gemm_bf16_mid: cannot reserve %d bytes of LDS: %s", bytes, hipGetErrorString(e));
      return 2;
    }
    configured = true;
  }
  const int steps_all = K / 128, per = (steps_all + shares - 1) / shares;
  const dim3 grid((N / 16 + NW - 1) / NW, (steps_all + per - 1) / per);
  gemm_bf16_mid_kernel<MT, AHEAD, NW, Scatter><<<grid, 64 * NW, bytes, stream>>>(x, w_tiles, bias, residual, out, out_dtype,
                                                                                 act, partial, M, N, K, per, sc);
  TNX_CHECK_LAUNCH("gemm_bf16_mid");
  return sum_shares(partial, bias, residual, out, out_dtype, act, M, N, (int)grid.y, left, stream);
}

// `shares` 0: chosen here (as many as give every compute unit a block at most, each with four steps of K or more,
// within the workspace); `ahead` 0: three steps in flight up to 64 rows, two beyond (what LDS holds).
static int gemm_bf16_mid(const void* x, const void* w_tiles, const float* bias, const float* residual, void* out, int out_dtype,
                         int act, int M, int N, int K, float* workspace, size_t workspace_floats, int shares, int ahead, int* left,
                         hipStream_t stream) {
  TNX_REQUIRE(M > 0 && M <= 128 && N > 0 && K > 0, "gemm_bf16_mid: takes 1 to 128 rows, got M=%d N=%d K=%d", M, N, K);
  TNX_REQUIRE(N % 16 == 0 && K % 128 == 0, "gemm_bf16_mid: the tile-ordered weight needs N a multiple of 16 and K "
              "of 128, got N=%d K=%d", N, K);
  TNX_REQUIRE(x && w_tiles && out && ((uintptr_t)x | (uintptr_t)w_tiles | (uintptr_t)workspace) % 16 == 0,
              "gemm_bf16_mid: operands must be there and 16-byte aligned");
  TNX_REQUIRE(out_dtype == TNX_F32 || out_dtype == TNX_BF16, "gemm_bf16_mid: the result is float32 or bfloat16");
  TNX_REQUIRE(shares >= 0 && (ahead == 0 || ahead == 2 || ahead == 3), "gemm_bf16_mid: bad shares, or steps ahead "
              "other than 2 and 3");
  const int blocks_n = (N / 16 + 3) / 4, steps_all = K / 128;
  if (shares == 0) {
    // a block a compute unit at most: blocks of one length in a ragged second round cost more than idle units
    shares = tnx_compute_units() / blocks_n;
    shares = max(1, min(shares, steps_all / 4));
  }
  shares = max(1, min(shares, steps_all));
  if (shares > 1) {
    const size_t room = workspace ? workspace_floats / ((size_t)M * N) : 0;
    if ((size_t)shares > room) shares = (int)max((size_t)1, room);
  }
  const bf16_t* xp = (const bf16_t*)x;
  const bf16_t* wp = (const bf16_t*)w_tiles;
  const int mt = (M + 15) / 16;
  if (ahead == 0) ahead = mt <= 4 ? 3 : 2;
  if (mt > 4 && ahead > 2) ahead = 2;               // what LDS holds
#define MID(MT, A) launch_mid<MT, A>(xp, wp, bias, residual, out, out_dtype, act, workspace, M, N, K, shares, left, stream)
#define MID_LOW(MT) return ahead == 2 ? MID(MT, 2) : MID(MT, 3)
#define MID_HIGH(MT) return MID(MT, 2)
  switch (mt) {
    case 1: MID_LOW(1);
    case 2: MID_LOW(2);
    case 3: MID_LOW(3);
    case 4: MID_LOW(4);
    case 5: MID_HIGH(5);
    case 6: MID_HIGH(6);
    case 7: MID_HIGH(7);
    default: MID_HIGH(8);
  }
#undef MID_HIGH
#undef MID_LOW
#undef MID
}

extern "C" int tnx_gemm_bf16_mid(const void* x, const void* w_tiles, const float* bias, const float* residual,
                                 void* out, int out_dtype, int act, int M, int N, int K, float* workspace,
                                 size_t workspace_floats, int shares, int ahead, hipStream_t stream) {
  return gemm_bf16_mid(x, w_tiles, bias, residual, out, out_dtype, act, M, N, K, workspace, workspace_floats, shares, ahead, nullptr,
                       stream);
}

// The same for 9 to 48 rows with a rounded result, or with queries, keys and values put in their places, and K whole: no sum
// follows, and what fills the chip is the number of waves a block has, two to four of 16 columns each: as many as leave every
// compute unit one block (`whole_waves`). A unit brings some 30 bytes a nanosecond from memory however many ask on it, so what
// counts is that all of them do: 10,240 columns of K 2,560 at 24 rows by blocks of one wave (640 blocks) to four (160) 17.2, 18.2,
// 14.6 and 17.0 us. Measured on weights that no cache holds, us, with what took them before (the few-rows kernel up to 24 rows
// or where the matrix is small, the vendor library beyond) / so, at 16, 24, 32 and 48 rows: 6,144 x 2,048 9.3 / 8.6, 11.1 / 9.8, 11.8 / 10.2,
// 13.5 / 11.9; 8,192 x 2,048 10.3 / 9.2, 12.0 / 10.3, 14.4 / 10.6, 15.1 / 12.6; 10,240 x 2,560 14.6 / 13.0, 20.8 / 14.6, 21.3 / 15.4, 20.7 / 19.8;
// 12,288 x 4,096 21.6 / 20.4, 28.4 / 21.5, 33.0 / 22.1, 28.2 / 25.2; 16,384 x 4,096 28.3 / 28.6, 32.0 / 29.8, 33.5 / 29.9, 35.6 / 32.6. Not for
// small matrices (24 rows 3,072 x 1,024 6.1 / 6.4: a chain of steps, where the few-rows kernel's waves share K) nor at 64 rows
// (12,288 x 4,096 27.5 / 29.4: the rows weigh as much as the weights), nor where one wave a block covers the columns (16 rows
// 4,096 x 4,096 10.4 / 12.8: the same chain); further lines stand with the rule (`HipOps._whole_product`).
template <typename Scatter>
static int launch_whole(const bf16_t* x, const bf16_t* w_tiles, const float* bias, void* out, int out_dtype, int act, int M, int N, int K,
                        int waves, const Scatter& sc, hipStream_t stream) {
#define WHOLE(MT, NW) launch_mid<MT, 3, NW, Scatter>(x, w_tiles, bias, nullptr, out, out_dtype, act, nullptr, M, N, K, 1, nullptr, stream, sc)
#define WHOLE_MT(MT) return waves == 2 ? WHOLE(MT, 2) : waves == 3 ? WHOLE(MT, 3) : WHOLE(MT, 4)
  if (M <= 32) WHOLE_MT(2);
  WHOLE_MT(3);
#undef WHOLE_MT
#undef WHOLE
}

static int whole_waves(int N) {
  const int units = tnx_compute_units(), tiles = N / 16;
  return max(2, min(4, (tiles + units - 1) / units));
}

static int whole_fits(const void* x, const void* w_tiles, int M, int N, int K, int waves) {
  TNX_REQUIRE(M > 0 && M <= 48 && N > 0 && N % 16 == 0 && K > 0 && K % 128 == 0 && (waves == 0 || (waves >= 2 && waves <= 4)),
              "gemm_bf16_whole: up to 48 rows, N a multiple of 16, K of 128, two to four waves; got M=%d N=%d K=%d waves=%d", M, N, K, waves);
  TNX_REQUIRE(x && w_tiles && ((uintptr_t)x | (uintptr_t)w_tiles) % 16 == 0, "gemm_bf16_whole: operands must be there and 16-byte aligned");
  return 0;
}

// `waves` 0: chosen here.
extern "C" int tnx_gemm_bf16_whole(const void* x, const void* w_tiles, const float* bias, void* out, int out_dtype, int act, int M, int N,
                                   int K, int waves, hipStream_t stream) {
  if (int rc = whole_fits(x, w_tiles, M, N, K, waves)) return rc;
  TNX_REQUIRE(out && (out_dtype == TNX_F32 || out_dtype == TNX_BF16), "gemm_bf16_whole: the result is float32 or bfloat16");
  return launch_whole((const bf16_t*)x, (const bf16_t*)w_tiles, bias, out, out_dtype, act, M, N, K, waves ? waves : whole_waves(N),
                      NoScatter{}, stream);
}

extern "C" int tnx_gemm_bf16_whole_qkv(const void* x, const void* w_tiles, const float* bias, int M, int K, const int* token_page,
                                       const int* token_off, void* q_out, void* k_pages, void* v_pages, float scale, int num_heads,
                                       int num_kv, int head_size, int page_size, int num_pages, int waves, const float* turn_a,
                                       const float* turn_b, const int* positions, int turn_rows, int page_pad, hipStream_t stream) {
  TNX_REQUIRE(num_heads > 0 && num_kv >= 0 && head_size > 0 && page_size > 0, "gemm_bf16_whole_qkv: bad sizes");
  const int nq = num_heads * head_size, nk = num_kv * head_size, N = nq + 2 * nk;
  if (int rc = whole_fits(x, w_tiles, M, N, K, waves)) return rc;
  QkvScatter sc{token_page, token_off, (bf16_t*)q_out, (bf16_t*)k_pages, (bf16_t*)v_pages, scale, nq, nk, head_size, num_kv, page_size, num_pages};
  if (int rc = qkv_turn(sc, turn_a, turn_b, positions, turn_rows, page_pad)) return rc;
  return launch_whole((const bf16_t*)x, (const bf16_t*)w_tiles, bias, nullptr, TNX_BF16, TNX_ACT_NONE, M, N, K,
                      waves ? waves : whole_waves(N), sc, stream);
}

// ------------------------------------------------------------------------------------- bfloat16, tiles

// out = act(x w^T + bias) + residual by tiles of 32 MI WM x 32 NI WN (`tiles.h`), K shared out over gridDim.y blocks where the
// result has too few tiles to give every compute unit one; the shares' float32 sums then go to `partial` and
// `gemm_mid_sum_kernel` adds them in their order. K is a multiple of 64, N of 8.
template <int MI, int NI, int ST, int WM, int WN>
__global__ void __launch_bounds__(64 * WM * WN) gemm_bf16_tiles_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                              const float* __restrict__ bias, const float* __restrict__ residual,
                                                              void* __restrict__ out, int out_dtype, int act,
                                                              float* __restrict__ partial, int M, int N, int K, int tiles_m,
                                                              int steps_per_share) {
  typedef Tile<MI, NI, ST, WM, WN> Products;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int at = by_xcd(blockIdx.x, gridDim.x);
  const int m0 = at % tiles_m * Products::TM, n0 = at / tiles_m * Products::TN;
  const int first = blockIdx.y * steps_per_share, steps = min(K / 64 - first, steps_per_share);
  Products t;
#pragma unroll
  for (int j = 0; j < Products::LA; ++j) {
    const int row = Products::x_row(j);
    t.xoff[j] = 2u * ((unsigned)min(m0 + row, M - 1) * (unsigned)K + Products::k_of(row));
  }
#pragma unroll
  for (int j = 0; j < Products::LB; ++j) {
    const int row = Products::w_row(j);
    t.woff[j] = 2u * ((unsigned)min(n0 + row, N - 1) * (unsigned)K + Products::k_of(row));
  }
  const int mw = m0 + Products::row0(), nw = n0 + Products::col0();
  // What the end adds is asked for before the products: there it would be one more time to reach memory, or two.
  float added[NI][16];
  f32x4 onto[Products::template out_count<float, 32 * NI>()];
  if (!partial) {
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n = nw + 32 * j + 8 * g + 4 * (int)((threadIdx.x >> 5) & 1);
#pragma unroll
        for (int e = 0; e < 4; ++e) added[j][4 * g + e] = bias ? bias[min(n + e, N - 1)] : 0.f;
      }
    if (residual) {
#pragma unroll
      for (int k = 0; k < Products::template out_count<float, 32 * NI>(); ++k)
        onto[k] = *(const f32x4*)(residual + (size_t)min(mw + Products::template out_row<float, 32 * NI>(k), M - 1) * N +
                                  min(nw + Products::template out_column<float, 32 * NI>(), N - 4));
    }
  }
  t.run(smem, x + 64 * first, w + 64 * first, steps);
  if (partial) {
    float* mine = partial + (size_t)blockIdx.y * M * N;
    t.template hand_out<float, 32 * NI>(
        smem, [&](int i, int j, int e, int, int) { return t.acc[i][j][e]; },
        [&](int r, int c, f32x4 chunk, int) {
          if (mw + r < M && nw + c < N) *(f32x4*)(mine + (size_t)(mw + r) * N + nw + c) = chunk;
        });
    return;
  }
  with_act(act, [&](auto activation) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) t.acc[i][j][e] = activation(t.acc[i][j][e] + added[j][e]);
  });
  auto value = [&](int i, int j, int e, int, int) { return t.acc[i][j][e]; };
  if (out_dtype == TNX_F32) {
    t.template hand_out<float, 32 * NI>(smem, value, [&](int r, int c, f32x4 chunk, int k) {
      if (residual) chunk += onto[k];
      if (mw + r < M && nw + c < N) *(f32x4*)((float*)out + (size_t)(mw + r) * N + nw + c) = chunk;
    });
  } else {
    t.template hand_out<bf16_t, 32 * NI>(smem, value, [&](int r, int c, f32x4 chunk, int) {
      if (mw + r < M && nw + c < N) *(f32x4*)((bf16_t*)out + (size_t)(mw + r) * N + nw + c) = chunk;
    });
  }
}

template <int MI, int NI, int ST, int WM, int WN>
static int launch_tiles(const bf16_t* x, const bf16_t* w, const float* bias, const float* residual, void* out, int out_dtype,
                        int act, float* partial, int M, int N, int K, int shares, int* left, hipStream_t stream) {
  constexpr int bytes = Tile<MI, NI, ST, WM, WN>::BYTES;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_bf16_tiles_kernel<MI, NI, ST, WM, WN>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    TNX_REQUIRE(e == hipSuccess, "gemm_bf16_tiles: cannot reserve %d bytes of LDS: %s", bytes, hipGetErrorString(e));
    configured = true;
  }
  const int tiles_m = (M + 32 * MI * WM - 1) / (32 * MI * WM), tiles_n = (N + 32 * NI * WN - 1) / (32 * NI * WN);
  const int per = (K / 64 + shares - 1) / shares;
  shares = (K / 64 + per - 1) / per;
  gemm_bf16_tiles_kernel<MI, NI, ST, WM, WN><<<dim3(tiles_m * tiles_n, shares), 64 * WM * WN, bytes, stream>>>(
      x, w, bias, residual, out, out_dtype, act, shares > 1 ? partial : nullptr, M, N, K, tiles_m, per);
  TNX_CHECK_LAUNCH("gemm_bf16_tiles");
  return sum_shares(partial, bias, residual, out, out_dtype, act, M, N, shares, left, stream);
}

// Which products these tiles take, and with which tile and how many shares of K (0: none, the vendor library).
// A unit pulls 57 bytes a nanosecond of lines that no cache holds, 70 where half of them come from its L2 (what hits waits in line behind
// what does not) and 135 to 160 where all do, however deep it asks; the weights of a model are in no cache. So at these sizes a tile's time
// is the bytes that its block brings, (TM + TN) 128 a step of 64 of K, and what counts is that the tiles are small and yet go round the
// units once. (More steps under way, K begun elsewhere by each block, a wave or loads that touch lines ahead and weights marked as
// read once were each measured to change 2 % or nothing.) `tiles_time`, us, is that: the bytes of the fullest unit, those of all blocks, a
// launch, and the sum of the shares. Tiles of 64 x 64 find two blocks a unit. Over 306 sizes of 33 to 768 rows it names the quickest of these
// tiles or one 2 % slower on average; on weights that no cache holds (16 matrices and more in turn), with bias and ReLU or the residual, us,
// the library / tiles of 64 x 64 and 128 x 128 alone / these:
//   333 rows 6,144 (columns) x 2,048 (K) 25.0 / 20.1 / 18.7, 8,192 x 2,048 23.4 / 20.9 / 19.8, 5,120 x 4,096 28.9 / - / 27.9;
//   200 rows 6,144 x 2,048 16.2 / 19.5 / 15.7, 8,192 x 2,048 17.7 / 20.1 / 16.2, 2,048 x 4,096 14.7 / - / 14.0;
//   100 rows 5,120 x 4,096 22.6 / - / 16.6, 2,048 x 8,192 19.3 / 16.2 / 14.4, 4,096 x 4,096 16.8 / - / 14.0; 64 rows 2,048 x 8,192 16.6 / 14.7 / 12.2;
//   512 rows 3,072 x 1,024 12.5 / 12.9 / 10.7, 7,680 x 2,560 31.8 / - / 28.5; 640 rows 2,048 x 4,096 25.6 / - / 23.0.
// The library keeps (library / tiles): matrices of many columns at up to 200 rows (128 rows 10,240 x 2,560 22.8 / 24.9, 100 rows 16,384 x 4,096
// 35.9 / 39.5; at 64 rows from 2^25 elements on), what would need more blocks than there are units (640 rows 8,192 x 2,048 26.4 / 40.8), many
// rows of few columns with K whole (768 rows 2,048 x 2,048 15.4 / 17.8, 512 rows 2,560 x 2,560 18.0 / 19.5), and K beyond 4,096 where tiles of
// 128 x 128 with their shares give half of the units a block or fewer, three quarters above 576 rows, or the rows are more than 704. A call of the
// library's takes the host some 13 us, a launch of ours 5, and short prompts are not recorded: a few per cent on the device are less than that.
// Tiles of 160 x 128 and 192 x 128, four waves and eight, were slower than the library where they would be taken (640 rows 8,192 x 2,048
// 31.3 and 26.7, 26.1), those of 96 x 64 no quicker than the others, and those of 96 x 96 only alone (333 rows 6,144 x 2,048 17.6 for 18.7; a prompt of
// 333 tokens of 1.3b 2,368 us with them and 2,363 without: one kernel fewer to fetch). Up to 32 rows half a tile would be padding, and other kernels stand ready.
enum { TILES_NONE = 0, TILES_64 = 1, TILES_128 = 2, TILES_64x128 = 3, TILES_96x128 = 4, TILES_MOST = 4 };

// (a product whose `blocks` of `rows` by `columns` make `per` steps of 64 of K each; `launch`: of the sum of the shares)
static float tiles_time(int rows, int columns, long long blocks, int M, int N, int per, int shares, int units, float launch) {
  const float block = 1e-3f * per * (rows + columns);
  const float sum = shares > 1 ? launch + 1.9e-6f * shares * M * N : 0.f;
  return 4.f + (blocks > units ? 2.16f : 1.6f) * block + 1.6e-3f * block * blocks + sum;
}

static int choose_tiles(int M, int N, int K, int& shares) {
  const int units = tnx_compute_units(), steps = K / 64;
  const long long large = (long long)((M + 127) / 128) * ((N + 127) / 128), matrix = (long long)N * K;
  shares = 1;
  if (M <= 32 || M > 768) return TILES_NONE;
  if (N > K && M <= 200 && matrix >= (M <= 64 ? 1ll << 25 : 3ll << 23)) return TILES_NONE;
  if (K > 4096) {
    if (K < 4ll * N || large > units) return TILES_NONE;
    const long long blocks = large * min(min(8ll, units / large), max(1ll, (long long)steps / 4));
    if (M > 128 && (M > 704 || 2 * blocks <= units || (M > 576 && 4 * blocks < 3 * units))) return TILES_NONE;
  }
  // (asked for every product of a prompt, whose host is what it waits for: no division twice, and none of 64 bits)
  int tile = TILES_NONE, most = 1, per[9] = {0, steps};
  while (most < 8 && steps >= 8 * (most + 1) && (long long)(most + 1) * M * N <= F32_SHARES_MOST) {
    ++most;
    per[most] = (steps + most - 1) / most;
  }
  // (behind a matrix that narrows stands a norm as a rule, whose launch adds the shares; behind one that widens the sum is a launch more for
  // the host and the device: 64 rows 6,144 x 2,048 in two shares take 13.6 us alone for 14.2, and a prompt of 64 tokens of 1.3b 2,558 for 2,435)
  const float launch = N > K ? 2.2f : 1.6f;
  float least = INFINITY;
  auto look = [&](int t, auto rows, auto columns) {
    constexpr int TM = decltype(rows)::value, TN = decltype(columns)::value;
    const long long tiles = (long long)((M + TM - 1) / TM) * ((N + TN - 1) / TN);
    for (int s = 1; s <= most; ++s) {
      if (4 * s * tiles > (t == TILES_64 && s == 1 ? 5 : 4) * units) break;
      // (shares that leave none for the last have their steps, and with fewer of them, already been asked for)
      if (s > 1 && per[s] * (s - 1) >= steps) continue;
      const float us = tiles_time(TM, TN, s * tiles, M, N, per[s], s, units, launch);
      if (us < least) least = us, tile = t, shares = s;
    }
  };
  look(TILES_64, std::integral_constant<int, 64>{}, std::integral_constant<int, 64>{});
  look(TILES_128, std::integral_constant<int, 128>{}, std::integral_constant<int, 128>{});
  look(TILES_64x128, std::integral_constant<int, 64>{}, std::integral_constant<int, 128>{});
  look(TILES_96x128, std::integral_constant<int, 96>{}, std::integral_constant<int, 128>{});
  // many rows of few columns, K whole
  if (K <= 4096 && (long long)M * K > 1ll << 20 && shares == 1 && (N <= K || (N <= 3072 && 2 * large <= units))) return TILES_NONE;
  return tile;
}

// Whether `tnx_gemm_bf16_tiles` is the way for a product (-1: it is not), and how many floats of workspace it then wants.
extern "C" int tnx_gemm_bf16_tiles_workspace(int M, int N, int K) {
  if (M <= 0 || N <= 0 || N % 8 || K <= 0 || K % 64) return -1;
  if ((long long)M * K >= (1ll << 31) || (long long)N * K >= (1ll << 31)) return -1;
  int shares = 1;
  if (choose_tiles(M, N, K, shares) == TILES_NONE) return -1;
  return shares > 1 ? shares * M * N : 0;
}

// `workspace`: as many floats as `tnx_gemm_bf16_tiles_workspace` names for the sizes. `tile`, `shares` 0: chosen here.
static int gemm_bf16_tiles(const void* x, const void* w, const float* bias, const float* residual, void* out, int out_dtype, int act,
                           int M, int N, int K, float* workspace, size_t workspace_floats, int tile, int shares, int* left,
                           hipStream_t stream) {
  TNX_REQUIRE(M > 0 && N > 0 && N % 8 == 0 && K > 0 && K % 64 == 0, "gemm_bf16_tiles: N in 8s and K in 64s, got M=%d N=%d K=%d", M, N, K);
  TNX_REQUIRE((long long)M * K < (1ll << 31) && (long long)N * K < (1ll << 31), "gemm_bf16_tiles: operands of 4 GB or more");
  TNX_REQUIRE(out_dtype == TNX_F32 || (out_dtype == TNX_BF16 && residual == nullptr), "gemm_bf16_tiles: a residual beside a float32 result");
  TNX_REQUIRE(((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)residual | (uintptr_t)workspace) % 16 == 0,
              "gemm_bf16_tiles: operands must be 16-byte aligned");
  TNX_REQUIRE(tile >= 0 && tile <= TILES_MOST && shares >= 0, "gemm_bf16_tiles: tiles 1 to %d", TILES_MOST);
  int chosen = 1;
  if (tile == 0) tile = choose_tiles(M, N, K, chosen);
  if (shares == 0) shares = chosen;
  if (shares > K / 64) shares = K / 64;
  if (shares > 1 && (workspace == nullptr || workspace_floats < (size_t)shares * M * N)) shares = 1;
  const bf16_t *xp = (const bf16_t*)x, *wp = (const bf16_t*)w;
#define TILES(MI, NI, WM, WN) return launch_tiles<MI, NI, 4, WM, WN>(xp, wp, bias, residual, out, out_dtype, act, workspace, M, N, K, shares, left, stream)
  switch (tile) {
    case TILES_128: TILES(2, 1, 2, 4);
    case TILES_64x128: TILES(2, 1, 1, 4);
    case TILES_96x128: TILES(3, 1, 1, 4);
    default: TILES(1, 1, 2, 2);
  }
#undef TILES
}

extern "C" int tnx_gemm_bf16_tiles(const void* x, const void* w, const float* bias, const float* residual, void* out,
                                   int out_dtype, int act, int M, int N, int K, float* workspace, size_t workspace_floats,
                                   int tile, int shares, hipStream_t stream) {
  return gemm_bf16_tiles(x, w, bias, residual, out, out_dtype, act, M, N, K, workspace, workspace_floats, tile, shares, nullptr, stream);
}

// A product of a float32 result onto a residual, by rows of some number (`way` 0), by tiles (1) or in float32 (2), whose shares of K
// stay apart where K is shared out: `left` says how many lie in `workspace`, one behind the other, for `tnx_shares_norm` or
// `tnx_gemm_shares_sum`; 1: `out` is the result.
extern "C" int tnx_gemm_left(int way, const void* x, const void* w, const float* bias, const float* residual, float* out, int M, int N,
                             int K, float* workspace, size_t workspace_floats, int tile, int shares, int* left, hipStream_t stream) {
  TNX_REQUIRE(way >= 0 && way <= 2 && left, "gemm_left: ways are 0 to 2");
  if (way == 0)
    return gemm_bf16_mid(x, w, bias, residual, out, TNX_F32, TNX_ACT_NONE, M, N, K, workspace, workspace_floats, shares, 0, left, stream);
  if (way == 1)
    return gemm_bf16_tiles(x, w, bias, residual, out, TNX_F32, TNX_ACT_NONE, M, N, K, workspace, workspace_floats, tile, shares, left, stream);
  return gemm_f32((const float*)x, (const float*)w, bias, residual, out, TNX_F32, TNX_ACT_NONE, M, N, K, workspace, workspace_floats, left,
                  stream);
}

// ------------------------------------------------------------------------------------- the vendor library
//
// out = act(x w^T + bias) + residual for many rows, as one call of hipBLASLt: bfloat16 operands, float32 sums,
// the bias (float32) and ReLU in the library's epilogue, and either a bfloat16 result or, for a product that
// ends in the residual sum, the float32 residual as the library's C matrix and a float32 result, so that such
// a product is never rounded to bfloat16 and no kernel of ours has to follow it. The library is the one the
// process has loaded already (torch brings it); its entry points are looked up at run time, so nothing here
// is linked against it.
// The library ranks its algorithms for a product by a model of its own. Up to TUNED_ROWS rows (decode batches,
// short portions of prompts) that ranking is often far off (128 x 4,096 over 16,384: first choice 116 us,
// sixth 68 us), so there the first six are timed once, on the operands of the first call, with the caches
// flushed before each run as a step finds them, and the quickest is kept. An algorithm is run only with all
// the workspace it asks for.
// Returns 0 when done, 1 on an error, 2 where this is not to be had (no library, an activation it has not,
// no algorithm that fits) and the caller goes another way, 3 when the algorithms are to be timed first and no
// memory to flush the caches with came along: the caller calls again with some.
#if __has_include(<hipblaslt/hipblaslt.h>)
#include <dlfcn.h>
#include <hipblaslt/hipblaslt.h>

#include <map>
#include <mutex>
#include <tuple>

namespace {
struct LibraryApi {
  decltype(&hipblasLtCreate) create = nullptr;
  decltype(&hipblasLtMatmulDescCreate) desc_create = nullptr;
  decltype(&hipblasLtMatmulDescSetAttribute) desc_set = nullptr;
  decltype(&hipblasLtMatrixLayoutCreate) layout_create = nullptr;
  decltype(&hipblasLtMatmulPreferenceCreate) pref_create = nullptr;
  decltype(&hipblasLtMatmulPreferenceSetAttribute) pref_set = nullptr;
  decltype(&hipblasLtMatmulPreferenceDestroy) pref_destroy = nullptr;
  decltype(&hipblasLtMatmulAlgoGetHeuristic) heuristic = nullptr;
  decltype(&hipblasLtMatmul) matmul = nullptr;
  int state = 0;                  // 0 not tried, 1 ready, -1 not to be had
};
struct LibraryPlan {
  hipblasLtMatmulDesc_t desc = nullptr;
  hipblasLtMatrixLayout_t w = nullptr, x = nullptr, c = nullptr;
  hipblasLtMatmulAlgo_t algo;
  size_t workspace = 0;
  bool usable = false;
};
struct LibraryCall {              // the operands of one product, as the library takes them
  const void *x, *w, *c;
  void* out;
  float beta;
  void* workspace;
  size_t workspace_bytes;
  hipStream_t stream;
};
constexpr int MAX_DEVICES = 64, CANDIDATES = 32, FEW_CANDIDATES = 6, TUNED_ROWS = 256;
LibraryApi library_api;
hipblasLtHandle_t library_handles[MAX_DEVICES] = {};
std::map<std::tuple<int, int, int, int, int>, LibraryPlan> library_plans;     // device, M, N, K, what follows
std::mutex library_mutex;

bool library_ready() {
  if (library_api.state != 0) return library_api.state > 0;
  library_api.state = -1;
  void* lib = dlopen("libhipblaslt.so.1", RTLD_NOW | RTLD_NOLOAD);      // the copy that is loaded, if one is
  if (!lib) lib = dlopen("libhipblaslt.so.1", RTLD_NOW);
  if (!lib) lib = dlopen("libhipblaslt.so", RTLD_NOW);
  if (!lib) return false;
#define TNX_LIBRARY_SYMBOL(field, name)                              \
  library_api.field = (decltype(library_api.field))dlsym(lib, name); \
  if (!library_api.field) return false;
  TNX_LIBRARY_SYMBOL(create, "hipblasLtCreate")
  TNX_LIBRARY_SYMBOL(desc_create, "hipblasLtMatmulDescCreate")
  TNX_LIBRARY_SYMBOL(desc_set, "hipblasLtMatmulDescSetAttribute")
  TNX_LIBRARY_SYMBOL(layout_create, "hipblasLtMatrixLayoutCreate")
  TNX_LIBRARY_SYMBOL(pref_create, "hipblasLtMatmulPreferenceCreate")
  TNX_LIBRARY_SYMBOL(pref_set, "hipblasLtMatmulPreferenceSetAttribute")
  TNX_LIBRARY_SYMBOL(pref_destroy, "hipblasLtMatmulPreferenceDestroy")
  TNX_LIBRARY_SYMBOL(heuristic, "hipblasLtMatmulAlgoGetHeuristic")
  TNX_LIBRARY_SYMBOL(matmul, "hipblasLtMatmul")
#undef TNX_LIBRARY_SYMBOL
  library_api.state = 1;
  return true;
}

hipblasStatus_t library_run(hipblasLtHandle_t handle, const LibraryPlan& p, const hipblasLtMatmulAlgo_t& algo,
                            const LibraryCall& call) {
  const float one = 1.f;
  return library_api.matmul(handle, p.desc, &one, call.w, p.w, call.x, p.x, &call.beta, call.c, p.c, call.out, p.c,
                            &algo, call.workspace, call.workspace_bytes, call.stream);
}

// Reads `bytes` of memory and keeps nothing: what the caches held before is pushed out by clean lines, as
// after the attention of a step, which has read the keys and values of every request.
__global__ void __launch_bounds__(256) library_flush_kernel(const float4* __restrict__ p, size_t n, float* sink) {
  float a = 0.f;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const float4 v = p[i];
    a += v.x + v.y + v.z + v.w;
  }
  if (a == 12345.678f) *sink = a;      // never true for memory that holds no such sum; keeps the loads alive
}

// Time in ms of a run of an algorithm with cold caches, the quickest of five (one run's time moves by more
// than the candidates differ when something else touches the device meanwhile), or a negative number if it
// cannot be run.
float library_time(hipblasLtHandle_t handle, const LibraryPlan& p, const hipblasLtMatmulAlgo_t& algo,
                   const LibraryCall& call, void* flush, size_t flush_bytes, hipEvent_t begin, hipEvent_t end) {
  for (int warm = 0; warm < 2; ++warm)
    if (library_run(handle, p, algo, call) != HIPBLAS_STATUS_SUCCESS) return -1.f;
  float best = -1.f;
  for (int run = 0; run < 5; ++run) {
    library_flush_kernel<<<2048, 256, 0, call.stream>>>((const float4*)flush, flush_bytes / 16, (float*)flush);
    if (hipGetLastError() != hipSuccess || hipEventRecord(begin, call.stream) != hipSuccess) return -1.f;
    if (library_run(handle, p, algo, call) != HIPBLAS_STATUS_SUCCESS) return -1.f;
    float ms = 0.f;
    if (hipEventRecord(end, call.stream) != hipSuccess || hipEventSynchronize(end) != hipSuccess ||
        hipEventElapsedTime(&ms, begin, end) != hipSuccess)
      return -1.f;
    if (best < 0.f || ms < best) best = ms;
  }
  return best;
}

// The plan of one product: descriptors and an algorithm. Row-major out[M][N] = x[M][K] w[N][K]^T is, in the
// library's column-major terms, D[N x M] = op_T(w as K x N) (x as K x M).
LibraryPlan make_plan(hipblasLtHandle_t handle, int M, int N, int K, const float* bias, bool relu, bool out_f32,
                      const LibraryCall& call, void* flush, size_t flush_bytes, int candidates) {
  LibraryPlan p;
  const LibraryApi& a = library_api;
  if (a.desc_create(&p.desc, HIPBLAS_COMPUTE_32F, HIP_R_32F) != HIPBLAS_STATUS_SUCCESS) return p;
  const hipblasOperation_t trans = HIPBLAS_OP_T, plain = HIPBLAS_OP_N;
  bool ok = a.desc_set(p.desc, HIPBLASLT_MATMUL_DESC_TRANSA, &trans, sizeof(trans)) == HIPBLAS_STATUS_SUCCESS &&
            a.desc_set(p.desc, HIPBLASLT_MATMUL_DESC_TRANSB, &plain, sizeof(plain)) == HIPBLAS_STATUS_SUCCESS;
  if (bias || relu) {
    const hipblasLtEpilogue_t epilogue =
        bias ? (relu ? HIPBLASLT_EPILOGUE_RELU_BIAS : HIPBLASLT_EPILOGUE_BIAS) : HIPBLASLT_EPILOGUE_RELU;
    ok = ok && a.desc_set(p.desc, HIPBLASLT_MATMUL_DESC_EPILOGUE, &epilogue, sizeof(epilogue)) == HIPBLAS_STATUS_SUCCESS;
  }
  if (bias) {
    const hipDataType bias_type = HIP_R_32F;
    const void* bias_ptr = bias;
    ok = ok && a.desc_set(p.desc, HIPBLASLT_MATMUL_DESC_BIAS_DATA_TYPE, &bias_type, sizeof(bias_type)) == HIPBLAS_STATUS_SUCCESS &&
         a.desc_set(p.desc, HIPBLASLT_MATMUL_DESC_BIAS_POINTER, &bias_ptr, sizeof(bias_ptr)) == HIPBLAS_STATUS_SUCCESS;
  }
  const hipDataType out_type = out_f32 ? HIP_R_32F : HIP_R_16BF;
  ok = ok && a.layout_create(&p.w, HIP_R_16BF, K, N, K) == HIPBLAS_STATUS_SUCCESS &&
       a.layout_create(&p.x, HIP_R_16BF, K, M, K) == HIPBLAS_STATUS_SUCCESS &&
       a.layout_create(&p.c, out_type, N, M, N) == HIPBLAS_STATUS_SUCCESS;
  if (!ok) return p;
  hipblasLtMatmulPreference_t pref = nullptr;
  if (a.pref_create(&pref) != HIPBLAS_STATUS_SUCCESS) return p;
  hipblasLtMatmulHeuristicResult_t found[CANDIDATES];
  int count = 0;
  const size_t room = call.workspace_bytes;
  if (a.pref_set(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &room, sizeof(room)) != HIPBLAS_STATUS_SUCCESS ||
      a.heuristic(handle, p.desc, p.w, p.x, p.c, p.c, pref, candidates, found, &count) != HIPBLAS_STATUS_SUCCESS)
    count = 0;
  a.pref_destroy(pref);
  int fits[CANDIDATES], n_fit = 0;
  for (int i = 0; i < count && i < candidates; ++i)
    if (found[i].state == HIPBLAS_STATUS_SUCCESS && found[i].workspaceSize <= room) fits[n_fit++] = i;
  if (n_fit == 0) return p;
  int pick = fits[0];
  if (flush && n_fit > 1) {
    hipEvent_t begin = nullptr, end = nullptr;
    if (hipEventCreate(&begin) == hipSuccess && hipEventCreate(&end) == hipSuccess) {
      float best = -1.f;
      for (int j = 0; j < n_fit; ++j) {
        const float t = library_time(handle, p, found[fits[j]].algo, call, flush, flush_bytes, begin, end);
        if (t >= 0.f && (best < 0.f || t < best)) {
          best = t;
          pick = fits[j];
        }
      }
    }
    if (begin) hipEventDestroy(begin);
    if (end) hipEventDestroy(end);
  }
  p.algo = found[pick].algo;
  p.workspace = found[pick].workspaceSize;
  p.usable = true;
  return p;
}
}  // namespace

extern "C" int tnx_gemm_library(const void* x, const void* w, const float* bias, const float* residual, void* out,
                                int out_dtype, int act, int M, int N, int K, void* workspace, size_t workspace_bytes,
                                void* flush, size_t flush_bytes, int tune, hipStream_t stream) {
  TNX_REQUIRE(M > 0 && N > 0 && K > 0 && N % 8 == 0 && K % 8 == 0, "gemm_library: bad sizes M=%d N=%d K=%d", M, N, K);
  TNX_REQUIRE(out_dtype == TNX_F32 || out_dtype == TNX_BF16, "gemm_library: the result is float32 or bfloat16");
  TNX_REQUIRE(residual == nullptr || out_dtype == TNX_F32, "gemm_library: a residual is added to a float32 result only");
  TNX_REQUIRE(((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)residual | (uintptr_t)bias |
               (uintptr_t)workspace) % 16 == 0,
              "gemm_library: operands must be 16-byte aligned");
  TNX_REQUIRE(out != (const void*)residual, "gemm_library: the sum is not made in place");
  if (act != TNX_ACT_NONE && act != TNX_ACT_RELU) return 2;
  if (act != TNX_ACT_NONE && residual) return 2;   // the library's ReLU comes after the residual sum, ours before it
  std::lock_guard<std::mutex> lock(library_mutex);
  if (!library_ready()) return 2;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= MAX_DEVICES) return 2;
  if (!library_handles[device] && library_api.create(&library_handles[device]) != HIPBLAS_STATUS_SUCCESS) {
    library_handles[device] = nullptr;
    return 2;
  }
  const LibraryCall call = {x, w, residual ? (const void*)residual : (const void*)out, out, residual ? 1.f : 0.f,
                            workspace, workspace_bytes, stream};
  const int what = (bias ? 1 : 0) | (residual ? 2 : 0) | (out_dtype == TNX_F32 ? 4 : 0) | (act == TNX_ACT_RELU ? 8 : 0);
  const auto key = std::make_tuple(device, M, N, K, what);
  auto it = library_plans.find(key);
  if (it == library_plans.end()) {
    // `tune` 1: up to TUNED_ROWS rows, and row counts that are multiples of 256 (the portions a token budget
    // cuts prompts into come again and again, and the ranking's first choice can be far off there too:
    // 2,048 x 9,216 over 36,864 with bias and ReLU, first choice 1.88 ms, the quickest of six about 1.1),
    // the first few of the ranking (more of it for the many rows, where the quickest was the ranking's
    // ninth or later: 2,048 x 4,096 over 16,384 with the float32 residual, first choice 246 us, the
    // nineteenth and twentieth 221 and 222, nothing quicker among 190); 2: every product, more of the ranking
    bool timed = tune >= 2 || (tune && (M <= TUNED_ROWS || M % 256 == 0));
    if (timed) {
      // nothing is timed inside a recording: the first choice of the library's ranking stands in there
      hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing(stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) timed = false;
    }
    if (timed && (flush == nullptr || flush_bytes == 0)) return 3;
    it = library_plans.emplace(key, make_plan(library_handles[device], M, N, K, bias, act == TNX_ACT_RELU,
                                              out_dtype == TNX_F32, call, timed ? flush : nullptr, flush_bytes,
                                              tune >= 2 || M > TUNED_ROWS ? CANDIDATES : FEW_CANDIDATES)).first;
  }
  const LibraryPlan& p = it->second;
  if (!p.usable || p.workspace > workspace_bytes) return 2;
  if (bias) {
    const void* bias_ptr = bias;
    if (library_api.desc_set(p.desc, HIPBLASLT_MATMUL_DESC_BIAS_POINTER, &bias_ptr, sizeof(bias_ptr)) !=
        HIPBLAS_STATUS_SUCCESS)
      return 2;
  }
  const hipblasStatus_t st = library_run(library_handles[device], p, p.algo, call);
  if (st != HIPBLAS_STATUS_SUCCESS) {
    tnx_set_error("gemm_library: the library refused the product (status %d) for M=%d N=%d K=%d", (int)st, M, N, K);
    return 1;
  }
  return 0;
}
#else
extern "C" int tnx_gemm_library(const void*, const void*, const float*, const float*, void*, int, int, int, int, int,
                                void*, size_t, void*, size_t, int, hipStream_t) {
  return 2;
}
#endif
