// Between the query/key/value projection and attention, for mixers whose queries and keys are normed over the
// whole projection, turned by halves, or whose values are blended or of a size of their own: one launch takes the
// float32 projections of a step's tokens to the queries (compute dtype) and to the tokens' places in the cache.
// Everything is float32 until the one rounding at the store.
#include "common.h"

TNX_DEFINE_ERROR_API

namespace {

struct PrepareArgs {
  const float* proj;        // [T, ld]: queries, keys, values side by side, bias added
  int ld;
  const float* q_weight;    // [H n] or null: no norm
  const float* k_weight;    // [G n]
  float eps;
  const float* freqs;       // [half] or null: no turning
  int half;
  int interleaved;
  const int* positions;     // [T]
  float scale;
  const float* mix_weight;  // [1] or null
  const float* first;       // [T, first_ld] or null: no blending
  long long first_ld;
  const int* token_page;    // [T]
  const int* token_offset;  // [T]
  void* q_out;              // [T, H D]
  void* k_pages;            // [pages, G, page, D]
  void* v_pages;            // [pages, G, D, page]
  long long page_stride;    // elements from one page to the next
  int num_pages, page_size;
  int heads, groups, n, v, d;
  int per_head;             // every head is normed by itself (the weights, if any, still one a projection element)
  int values_at;            // the column of a row where the values begin (behind the keys, or the keys' own)
  const float* head_scale;  // [H] or null: a query head's elements times its number, beside `scale`
  float temp_coef;          // the queries of position p times 1 + temp_coef ln(floor((p + 1) / temp_every) + 1)
  int temp_every;           // 0: not
  int tokens;
  int fours;                // four neighbouring elements of the queries and keys a thread
};

typedef float f32x4p __attribute__((ext_vector_type(4)));
template <typename T>
struct Four {
  typedef T type __attribute__((ext_vector_type(4)));
};

// what the token's queries are multiplied by, beside a head's own number
__device__ __forceinline__ float query_scale(const PrepareArgs& a, int t) {
  if (a.temp_every <= 0) return a.scale;
  return a.scale * (1.f + a.temp_coef * logf((float)((a.positions[t] + 1) / a.temp_every + 1)));
}

// Element `e` of head `head` of a normed projection, turned by the token's position. `x` points at the
// projection's first head, `w` at its norm weight (or null), `r` is the factor of the norm.
__device__ __forceinline__ float turned(const float* x, const float* w, float r, int head, int e, const PrepareArgs& a,
                                        const float* cosines, const float* sines) {
  const int at = head * a.n + e;
  const float own = x[at] * r * (w ? w[at] : 1.f);
  if (a.freqs == nullptr || e >= 2 * a.half) return own;
  int i, other;
  bool first;
  if (a.interleaved) {
    i = e >> 1;
    first = (e & 1) == 0;
    other = first ? e + 1 : e - 1;
  } else {
    first = e < a.half;
    i = first ? e : e - a.half;
    other = first ? e + a.half : e - a.half;
  }
  const int oat = head * a.n + other;
  const float mate = x[oat] * r * (w ? w[oat] : 1.f);
  const float s = sines[i], c = cosines[i];
  // the pair (u, v) becomes (u c - v s, v c + u s)
  return first ? own * c - mate * s : own * c + mate * s;
}

// Elements `e` to `e + 3` of head `head`, likewise (`fours`: turned by halves of a multiple of four elements, or not at all).
__device__ __forceinline__ f32x4p turned4(const float* x, const float* w, float r, int head, int e, const PrepareArgs& a,
                                          const float* cosines, const float* sines) {
  const int at = head * a.n + e;
  f32x4p own = *(const f32x4p*)(x + at) * r;
  if (w) own *= *(const f32x4p*)(w + at);
  if (a.freqs == nullptr || e >= 2 * a.half) return own;
  const bool first = e < a.half;
  const int i = first ? e : e - a.half, oat = first ? at + a.half : at - a.half;
  f32x4p mate = *(const f32x4p*)(x + oat) * r;
  if (w) mate *= *(const f32x4p*)(w + oat);
  const f32x4p s = *(const f32x4p*)(sines + i), c = *(const f32x4p*)(cosines + i);
  return first ? own * c - mate * s : own * c + mate * s;
}

// What a value's place in the cache holds: element `i` of `groups * d` of token `t`.
__device__ __forceinline__ float value_of(const PrepareArgs& a, int t, int i, float lam) {
  const int g = i / a.d, e = i - g * a.d;
  if (e >= a.v) return 0.f;
  const float val = a.proj[(size_t)t * a.ld + a.values_at + g * a.v + e];
  return a.first != nullptr ? (1.f - lam) * val + lam * a.first[(size_t)t * a.first_ld + g * a.v + e] : val;
}

// Values of many tokens: a page holds an element's values of all its tokens side by side, so 64 tokens of 64 elements go
// through LDS and a wave stores 64 tokens of one element. A token at a time every
// value is a store of two bytes of its own. A thread asks for all of its 16 elements before it uses one: asked for one after the
// other they were the launch's longest chain (396 tokens, 32 + 2 x 8 heads of 64, blended values 12.8 us, 7.1 so; 2,048 of 128 29.1 and 27.5).
template <typename T>
__device__ __forceinline__ void values_by_tiles(const PrepareArgs& a, int block, int blocks, float (*tile)[65]) {
  const int count = a.groups * a.d, across = (count + 63) / 64, tiles = (a.tokens + 63) / 64 * across;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float lam = a.first != nullptr ? a.mix_weight[0] : 0.f;
  for (int at = block; at < tiles; at += blocks) {
    const int t0 = at / across * 64, i0 = at % across * 64;
    const int mine = t0 + lane;
    const int page = mine < a.tokens ? a.token_page[mine] : -1, off = mine < a.tokens ? a.token_offset[mine] : 0;
    // (from places that are valid whatever a lane's token and element are, so that all are on their way at once)
    const int i = min(i0 + lane, count - 1), g = i / a.d, e = i - g * a.d, column = g * a.v + min(e, a.v - 1);
    float val[16], blend[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) val[k] = a.proj[(size_t)min(t0 + wave + 4 * k, a.tokens - 1) * a.ld + a.values_at + column];
    if (a.first != nullptr) {
#pragma unroll
      for (int k = 0; k < 16; ++k) blend[k] = a.first[(size_t)min(t0 + wave + 4 * k, a.tokens - 1) * a.first_ld + column];
#pragma unroll
      for (int k = 0; k < 16; ++k) val[k] = (1.f - lam) * val[k] + lam * blend[k];
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) tile[lane][wave + 4 * k] = e < a.v ? val[k] : 0.f;
    __syncthreads();
    if (page >= 0 && page < a.num_pages) {         // the host checks that every token has a page
      T* vp = (T*)a.v_pages + (size_t)page * a.page_stride + off;
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int i = wave + 4 * k;
        if (i0 + i < count) vp[(size_t)(i0 + i) * a.page_size] = from_f32<T>(tile[i][lane]);
      }
    }
    __syncthreads();
  }
}

// Latency bounds it for few tokens, memory for many (2,048 tokens of 32 + 2 x 8 heads of 128: 76 MB). Elements one by one
// and values a token at a time took 5.7 us for 8 tokens and 44.8 for 2,048; four at a time and by tiles 4.5 and 25.6.
// grid: (tokens, 3, shares), values first: a block takes a share of a token's queries, keys or values; each of the three needs nothing
// of the other two. (A norm over the whole projection is summed up by every block that shares it.)
template <typename T, bool TILED>
__global__ void __launch_bounds__(256) qkv_prepare_kernel(PrepareArgs a) {
  __shared__ float scratch[4];
  __shared__ __attribute__((aligned(16))) float cosines[128], sines[128];       // of the token's angles, once for all heads
  __shared__ float tile[TILED ? 64 : 1][65];
  const int t = blockIdx.x, part = 2 - blockIdx.y, share = blockIdx.z, shares = gridDim.z;
  if (TILED && part == 2) return values_by_tiles<T>(a, t + a.tokens * share, a.tokens * shares, tile);
  const float* row = a.proj + (size_t)t * a.ld;
  const int nq = a.heads * a.n, nk = a.groups * a.n;
  const int page = a.token_page[t], off = a.token_offset[t];
  if (part > 0 && (page < 0 || page >= a.num_pages)) return;       // the host checks that every token has a page
  if (part == 2) {
    T* vp = (T*)a.v_pages + (size_t)page * a.page_stride;
    const float lam = a.first != nullptr ? a.mix_weight[0] : 0.f;
    for (int i = threadIdx.x + 256 * share; i < a.groups * a.d; i += 256 * shares)
      vp[(size_t)i * a.page_size + off] = from_f32<T>(value_of(a, t, i, lam));
    return;
  }
  const float scale = part == 0 ? query_scale(a, t) : 1.f;
  if (a.freqs != nullptr) {
    const float pos = (float)a.positions[t];
    for (int i = threadIdx.x; i < a.half; i += 256) sincosf(pos * a.freqs[i], &sines[i], &cosines[i]);
  }
  // queries (part 0) or keys (part 1): the norm over the whole projection, then head by head
  const float* x = part == 0 ? row : row + nq;
  const float* w = part == 0 ? a.q_weight : a.k_weight;
  const int count = part == 0 ? nq : nk, heads = part == 0 ? a.heads : a.groups;
  if (a.per_head) {
    // a wave a head: the head's sum of squares over its lanes, then its elements
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();       // the token's sines and cosines are there
    T* kp = part == 1 ? (T*)a.k_pages + (size_t)page * a.page_stride : nullptr;
    T* q_out = part == 0 ? (T*)a.q_out + (size_t)t * a.heads * a.d : nullptr;
    for (int head = wave + 4 * share; head < heads; head += 4 * shares) {
      float s = 0.f;
      for (int e = lane; e < a.n; e += 64) s += x[head * a.n + e] * x[head * a.n + e];
      const float r = 1.f / sqrtf(wave_sum(s) / (float)a.n + a.eps);
      for (int e = lane; e < a.d; e += 64) {
        const float val = e < a.n ? turned(x, w, r, head, e, a, cosines, sines) : 0.f;
        if (part == 0)
          q_out[head * a.d + e] = from_f32<T>(val * (a.head_scale ? scale * a.head_scale[head] : scale));
        else
          kp[((size_t)head * a.page_size + off) * a.d + e] = from_f32<T>(val);
      }
    }
    return;
  }
  float norm = 1.f;
  if (w != nullptr) {
    float s = 0.f;
    if (a.fours) {
      for (int i = threadIdx.x; i < count / 4; i += 256) {
        const f32x4p z = ((const f32x4p*)x)[i];
        s += z[0] * z[0] + z[1] * z[1] + z[2] * z[2] + z[3] * z[3];
      }
    } else {
      for (int i = threadIdx.x; i < count; i += 256) s += x[i] * x[i];
    }
    s = block_sum<4>(s, scratch);
    norm = 1.f / sqrtf(s / (float)count + a.eps);
  }
  __syncthreads();
  if (a.fours) {
    typedef typename Four<T>::type four;
    T* out = part == 0 ? (T*)a.q_out + (size_t)t * a.heads * a.d
                       : (T*)a.k_pages + (size_t)page * a.page_stride + (size_t)off * a.d;
    const size_t apart = part == 0 ? a.d : (size_t)a.page_size * a.d;          // from a head to the next
    const int per = a.d / 4;
    for (int i = threadIdx.x + 256 * share; i < heads * per; i += 256 * shares) {
      const int head = i / per, e = 4 * (i - head * per);
      f32x4p val = {0.f, 0.f, 0.f, 0.f};
      if (e < a.n) val = turned4(x, w, norm, head, e, a, cosines, sines) * (part == 0 && a.head_scale ? scale * a.head_scale[head] : scale);
      four o;
#pragma unroll
      for (int c = 0; c < 4; ++c) o[c] = from_f32<T>(val[c]);
      *(four*)(out + head * apart + e) = o;
    }
    return;
  }
  if (part == 0) {
    T* q_out = (T*)a.q_out + (size_t)t * a.heads * a.d;
    for (int i = threadIdx.x + 256 * share; i < heads * a.d; i += 256 * shares) {
      const int head = i / a.d, e = i - head * a.d;
      q_out[i] = from_f32<T>(e < a.n ? turned(x, w, norm, head, e, a, cosines, sines) *
                                           (a.head_scale ? scale * a.head_scale[head] : scale)
                                     : 0.f);
    }
  } else {
    T* kp = (T*)a.k_pages + (size_t)page * a.page_stride;
    for (int i = threadIdx.x + 256 * share; i < heads * a.d; i += 256 * shares) {
      const int g = i / a.d, e = i - g * a.d;
      kp[((size_t)g * a.page_size + off) * a.d + e] = from_f32<T>(e < a.n ? turned(x, w, norm, g, e, a, cosines, sines) : 0.f);
    }
  }
}

}  // namespace

// `longest`: the tokens of the step's longest run, or fewer where 64 of them or `tokens` below 100 say enough.
extern "C" int tnx_qkv_prepare(const float* proj, int ld, const float* q_weight, const float* k_weight, float eps,
                               const float* freqs, int half, int interleaved, const int* positions, float scale,
                               const float* mix_weight, const float* first, long long first_ld, const int* token_page,
                               const int* token_offset, void* q_out, void* k_pages, void* v_pages, long long page_stride,
                               int num_pages, int page_size, int dtype, int tokens, int heads, int groups, int n, int v,
                               int d, int per_head, int values_at, const float* head_scale, float temp_coef, int temp_every,
                               int longest, hipStream_t stream) {
  TNX_REQUIRE(tokens >= 0 && heads > 0 && groups > 0 && n > 0 && v > 0, "qkv_prepare: bad sizes");
  TNX_REQUIRE(d >= n && d >= v, "qkv_prepare: cached heads of %d elements do not hold %d and %d", d, n, v);
  if (values_at < 0) values_at = heads * n + groups * n;
  TNX_REQUIRE(ld >= heads * n + groups * n && ld >= values_at + groups * v,
              "qkv_prepare: rows of %d elements do not hold the keys and the values at column %d", ld, values_at);
  TNX_REQUIRE(freqs == nullptr || (2 * half <= n && half <= 128), "qkv_prepare: %d turned elements in heads of %d", 2 * half, n);
  TNX_REQUIRE((q_weight == nullptr) == (k_weight == nullptr), "qkv_prepare: both norm weights or none");
  TNX_REQUIRE((first == nullptr) || (mix_weight != nullptr && first_ld >= groups * v), "qkv_prepare: blending needs its weight");
  TNX_REQUIRE(page_stride >= (long long)groups * d * page_size, "qkv_prepare: pages closer than a page's elements");
  TNX_REQUIRE(dtype == TNX_F32 || dtype == TNX_BF16, "qkv_prepare: dtype %d", dtype);
  if (tokens == 0) return 0;
  PrepareArgs a{proj, ld, q_weight, k_weight, eps, freqs, half, interleaved, positions, scale, mix_weight, first, first_ld,
                token_page, token_offset, q_out, k_pages, v_pages, page_stride, num_pages, page_size, heads, groups, n, v, d,
                per_head, values_at, head_scale, temp_coef, temp_every, tokens, 0};
  // four neighbours at a time where heads, rows and places allow it (a row's start is its keys' start and a head's as well)
  const uintptr_t ends = (uintptr_t)proj | (uintptr_t)q_weight | (uintptr_t)k_weight | (uintptr_t)q_out | (uintptr_t)k_pages;
  a.fours = n % 4 == 0 && d % 4 == 0 && ld % 4 == 0 && page_stride % 4 == 0 && ends % 16 == 0 &&
            (freqs == nullptr || (!interleaved && half % 4 == 0));
  // few tokens: a token's heads over several blocks
  int shares = 1;
  while (shares < 8 && 6ll * tokens * shares <= tnx_compute_units() && heads * d >= 1024 * shares) shares *= 2;
  const dim3 grid(tokens, 3, shares);
  // Values by tiles where a tile's tokens lie side by side in their pages, from runs of 64 tokens on, and where there is a block
  // for every tile: from 100 tokens on, and from 48 tiles, fewer leave most units without one. us, a token at a time / by
  // tiles, 32 query heads, one run: 8 heads of 64, 256 tokens (32 tiles) 5.9 / 6.7, 400 (56) 6.8 / 6.8, 2,048 19.4 / 15.1; 8 of
  // 128, 160 (48) 7.5 / 6.9, 256 (64) 8.2 / 7.2, 2,048 30.6 / 25.6; 32 of 128, 80 (128) 8.4 / 9.4, 100 9.9 / 10.0, 128 10.4 / 7.1,
  // 2,048 81.7 / 40.4. Requests of one token each, whose places are a page apart: 1 (64 tiles, 8 blocks) 4.3 / 16.9, 64 10.1 /
  // 12.5, 200 17.5 / 20.4, 400 31.1 / 32.6.
  const bool tiled = longest >= 64 && tokens >= 100 && ((long long)tokens + 63) / 64 * (((long long)groups * d + 63) / 64) >= 48;
  if (dtype == TNX_F32) {
    if (tiled) qkv_prepare_kernel<float, true><<<grid, 256, 0, stream>>>(a);
    else qkv_prepare_kernel<float, false><<<grid, 256, 0, stream>>>(a);
  } else {
    if (tiled) qkv_prepare_kernel<bf16_t, true><<<grid, 256, 0, stream>>>(a);
    else qkv_prepare_kernel<bf16_t, false><<<grid, 256, 0, stream>>>(a);
  }
  TNX_CHECK_LAUNCH("qkv_prepare");
  return 0;
}
