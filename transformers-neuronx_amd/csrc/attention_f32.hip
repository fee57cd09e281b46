// Attention of the float32 engine over the paged cache, every product and sum in float32:
//   prompt   queries of runs of several tokens, on the float32 matrix instructions (32x32x2)
//   decode   one query a request: the keys and values read once, plain FMA
// Head sizes in steps of 16 up to 128; others stay with `attention_any` (attention.hip), one wave a query.
// Keys [pages, kv_heads, page_size, head_size], values [pages, kv_heads, head_size, page_size], pages of any
// multiple of 16 tokens.
#include "common.h"

TNX_DEFINE_ERROR_API

namespace {

struct F32Attention {
  const float* q;
  const float* k_pages;
  const float* v_pages;
  const int* run_start;
  const int* cached_lens;
  const int* table;
  const int* tile_run;
  const int* tile_start;
  const int* decode_runs;
  float* out;
  int table_width, page_size, num_pages, num_heads, num_kv, window, num_tiles;
  size_t page_stride;    // elements from one page to the next
};

// The page of position `key` of the request whose row of the block table is `tab`; 0 where it holds none (`held` false).
__device__ __forceinline__ int page_of(const F32Attention& a, const int* tab, int key, bool& held) {
  const int page = tab[min(key / a.page_size, a.table_width - 1)];
  held = page >= 0 && page < a.num_pages;
  return held ? page : 0;
}

__device__ __forceinline__ float other_half(float x) {      // of lane ^ 32
  unsigned lo, hi;
  swap_halves(__float_as_uint(x), lo, hi);
  return __uint_as_float((threadIdx.x & 32) ? lo : hi);
}

// 32 queries of one head a block; its four waves take the blocks of 32 keys in turn and meet in LDS at the end, so that a
// short prompt's few tiles have four times the waves (300 tokens of 32 heads: 320 tiles on 256 compute units).
// S^T = K Q^T: a lane's 16 results belong to one query (lane % 32) and to the keys 8 g + 4 (lane / 32) + c of element
// 4 g + c, which is just what the second product O^T = V^T P^T wants of its right operand (lane / 32 is the k of a
// 32x32x2 product): the weights never leave their registers. Keys and values come straight from the cache, 16 bytes a
// lane, and need no LDS: a wave's 64 products of 64 cycles over a block of 32 keys (head size 64) are paid for with
// 16 KB of reads, 4 bytes a cycle. What bounds it is the rate of the float32 matrix instructions.
// Measured at runs of 300 and 101 tokens, 32 heads of 64: 27 us, against 362 with one wave a query and plain FMA.
// The block's number counts heads first, then tiles, then the 32 queries within a tile: blocks go round the XCDs in their
// order, and of a short run only the first 32 queries are there. With these first only every fourth block had work, all on
// two XCDs of eight: 8 runs of 2 tokens, 32 heads of 80, 30.4 us, 10.7 so.
template <int HD>
__global__ void __launch_bounds__(256, HD <= 64 ? 2 : 1)
attention_prompt_f32_kernel(F32Attention a) {
  constexpr int QS = HD / 8;                       // steps of 8 elements of the first product
  constexpr int HT = (HD + 31) / 32;               // tiles of 32 elements of the second
  constexpr int ROW = HD + 4;
  extern __shared__ float merged[];                // [4][32][ROW], then m and l [4][32] each
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l32 = lane & 31, half = lane >> 5;
  const int h = blockIdx.x % a.num_heads, kvh = h / (a.num_heads / a.num_kv);
  const int of_all = blockIdx.x / a.num_heads, tile = of_all % a.num_tiles;
  const int run = a.tile_run[tile];
  const int first = a.run_start[run], count = a.run_start[run + 1] - first;
  const int q0 = a.tile_start[tile] + 32 * (of_all / a.num_tiles);
  if (q0 >= count) return;                         // the whole block
  const int cached = a.cached_lens[run];
  const int* tab = a.table + (size_t)run * a.table_width;
  const size_t nq = (size_t)a.num_heads * HD;
  const int my_q = min(q0 + l32, count - 1);
  const int pos = cached + my_q;                   // of this lane's query
  const int last = cached + min(q0 + 31, count - 1);
  const int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  const int first_lo = a.window > 0 ? max(0, cached + q0 - a.window + 1) : 0;

  f32x4 q[QS];
#pragma unroll
  for (int s = 0; s < QS; ++s) q[s] = *(const f32x4*)(a.q + (size_t)(first + my_q) * nq + h * HD + 8 * s + 4 * half);

  f32x16 o[HT];
#pragma unroll
  for (int t = 0; t < HT; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
  float m = -INFINITY, l = 0.f;

  for (int key0 = (first_lo / 32 + wave) * 32; key0 <= last; key0 += 128) {
    bool held;
    const int page = page_of(a, tab, key0 + l32, held);
    const float* kp = a.k_pages + (size_t)page * a.page_stride +
                      ((size_t)kvh * a.page_size + (key0 + l32) % a.page_size) * HD + 4 * half;
    const float* vp[4];
    unsigned v_held = 0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int key = key0 + 8 * g + 4 * half;     // four keys of one page: pages are multiples of 16 tokens
      bool vh;
      const int vpage = page_of(a, tab, key, vh);
      v_held |= (unsigned)vh << g;
      vp[g] = a.v_pages + (size_t)vpage * a.page_stride + (size_t)kvh * HD * a.page_size + key % a.page_size;
    }
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.f;
    f32x4 kk[QS];
#pragma unroll
    for (int i = 0; i < QS; ++i) kk[i] = *(const f32x4*)(kp + 8 * i);
    f32x4 v[HT][4];
#pragma unroll
    for (int t = 0; t < HT; ++t) {
      const size_t d = (size_t)min(32 * t + l32, HD - 1) * a.page_size;     // rows beyond the head are dropped
#pragma unroll
      for (int g = 0; g < 4; ++g) v[t][g] = *(const f32x4*)(vp[g] + d);
    }
#pragma unroll
    for (int i = 0; i < QS; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kk[i][c], q[i][c], s, 0, 0, 0);

    // whole: every key of the block is there and is seen by every query of the tile
    const bool whole = key0 + 31 <= cached + q0 && key0 >= (a.window > 0 ? last - a.window + 1 : 0) &&
                       __all(v_held == 15);
    if (!whole) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int key = key0 + 8 * (e >> 2) + 4 * half + (e & 3);
        if (key > pos || key < lo || !((v_held >> (e >> 2)) & 1)) s[e] = -INFINITY;
      }
      // values at places that were never written must not meet a weight of zero as NaN
#pragma unroll
      for (int t = 0; t < HT; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int key = key0 + 8 * g + 4 * half + c;
            if (key > last || key < first_lo || !((v_held >> g) & 1)) v[t][g][c] = 0.f;
          }
    }
    float top = s[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) top = fmaxf(top, s[e]);
    const float m_new = fmaxf(m, fmaxf(top, other_half(top)));
    float p[16], sum = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      p[e] = s[e] == -INFINITY ? 0.f : expf(s[e] - m_new);
      sum += p[e];
    }
    sum += other_half(sum);
    const float alpha = m == m_new ? 1.f : expf(m - m_new);      // (no key seen so far: both are -inf)
    l = l * alpha + sum;
    m = m_new;
    bool odd = false;      // a value that is no number, at a key that some query of the tile does not see
    if (!whole) {
#pragma unroll
      for (int t = 0; t < HT; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int c = 0; c < 4; ++c) odd |= !(fabsf(v[t][g][c]) <= 3.402823466e38f);
    }
#pragma unroll
    for (int t = 0; t < HT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[t][e] *= alpha;
    if (!whole && __any(odd)) {
      // such a value may reach the queries that see its key and no others: key by key
#pragma unroll 1
      for (int j = 0; j < 32; ++j) {
        const int key = key0 + j;
        float pj = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (((e >> 2) << 1) + half == j >> 2 && (e & 3) == (j & 3)) pj = p[e];
        const float beside = other_half(pj);
        if (((j >> 2) & 1) != half) pj = beside;
        bool vh;
        const int vpage = page_of(a, tab, key, vh);
        const float* vj = a.v_pages + (size_t)vpage * a.page_stride + (size_t)kvh * HD * a.page_size + key % a.page_size;
        if (!vh || key > pos || key < lo) continue;
#pragma unroll
        for (int t = 0; t < HT; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int d = 32 * t + 8 * (e >> 2) + 4 * half + (e & 3);
            o[t][e] = fmaf(pj, vj[(size_t)min(d, HD - 1) * a.page_size], o[t][e]);
          }
      }
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int t = 0; t < HT; ++t)
            o[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[t][g][c], p[4 * g + c], o[t], 0, 0, 0);
    }
  }

  // the four waves' results: each is scaled to the highest of their maxima and they are added in their order
  float* ms = merged + 4 * 32 * ROW;
  float* ls = ms + 128;
  if (half == 0) {
    ms[wave * 32 + l32] = m;
    ls[wave * 32 + l32] = l;
  }
#pragma unroll
  for (int t = 0; t < HT; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      if (32 * t + 8 * g + 4 * half < HD)
        *(f32x4*)(merged + (size_t)(wave * 32 + l32) * ROW + 32 * t + 8 * g + 4 * half) =
            (f32x4){o[t][4 * g], o[t][4 * g + 1], o[t][4 * g + 2], o[t][4 * g + 3]};
  __syncthreads();
  for (int i = threadIdx.x; i < 32 * HD; i += 256) {
    const int r = i / HD, d = i % HD;
    if (q0 + r >= count) break;
    float top = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) top = fmaxf(top, ms[w * 32 + r]);
    float sum = 0.f, v = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float mw = ms[w * 32 + r];
      // (a wave that saw no key of this query brings sums of zero; one whose scores are no numbers, which a maximum passes
      // over, brings sums that are none either: no wave is left out)
      const float f = mw == top ? 1.f : expf(mw - top);
      sum += f * ls[w * 32 + r];
      v += f * merged[(size_t)(w * 32 + r) * ROW + d];
    }
    a.out[(size_t)(first + q0 + r) * nq + h * HD + d] = v * (1.f / sum);
  }
}

// One query: a block of eight waves a (request, head), a wave 64 keys at a time. For the scores a lane takes a key and
// reads its row 16 bytes at a time; for the weighted values sixteen lanes take the 64 keys of an element, four each, so
// that a lane's sums need no exchange before the last key. Keys and values of a chunk are asked for together. What bounds
// it at the contexts of a conversation is the time to reach memory, once a chunk. Measured at 3 requests of 60 to 76
// tokens, 16 heads of 64: 7.8 us, against 24.3 with one wave a query.
template <int HD>
__global__ void __launch_bounds__(512)
attention_decode_f32_kernel(F32Attention a) {
  constexpr int WAVES = 8;
  constexpr int H4 = HD / 4;
  __shared__ __attribute__((aligned(16))) float qs[HD];
  __shared__ __attribute__((aligned(16))) float ps[WAVES][64];
  __shared__ float os[WAVES][HD], ms[WAVES], ls[WAVES];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int run = a.decode_runs[blockIdx.x], h = blockIdx.y, kvh = h / (a.num_heads / a.num_kv);
  const int token = a.run_start[run], pos = a.cached_lens[run];
  const int* tab = a.table + (size_t)run * a.table_width;
  const size_t at = (size_t)token * a.num_heads * HD + h * HD;
  for (int d = threadIdx.x; d < HD; d += 512) qs[d] = a.q[at + d];
  __syncthreads();
  const int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  float m = -INFINITY, l = 0.f, acc[H4];
#pragma unroll
  for (int i = 0; i < H4; ++i) acc[i] = 0.f;
  for (int key0 = (lo / 64 + wave) * 64; key0 <= pos; key0 += 64 * WAVES) {
    const int key = key0 + lane, vkey = key0 + 4 * (lane & 15);
    bool held, v_held;
    const int page = page_of(a, tab, min(key, pos), held), vpage = page_of(a, tab, min(vkey, pos), v_held);
    const float* kp = a.k_pages + (size_t)page * a.page_stride +
                      ((size_t)kvh * a.page_size + min(key, pos) % a.page_size) * HD;
    // (four keys of one page: positions beyond the last are read from the last one's group of four)
    const float* vp = a.v_pages + (size_t)vpage * a.page_stride +
                      ((size_t)kvh * HD + (lane >> 4)) * a.page_size + (min(vkey, pos) & ~3) % a.page_size;
    f32x4 kk[H4], v[H4];
#pragma unroll
    for (int i = 0; i < H4; ++i) kk[i] = *(const f32x4*)(kp + 4 * i);
#pragma unroll
    for (int i = 0; i < H4; ++i) v[i] = *(const f32x4*)(vp + (size_t)4 * i * a.page_size);
    f32x4 s4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < H4; ++i) {
      const f32x4 qv = *(const f32x4*)(qs + 4 * i);
#pragma unroll
      for (int c = 0; c < 4; ++c) s4[c] = fmaf(kk[i][c], qv[c], s4[c]);
    }
    const bool seen = key >= lo && key <= pos && held;
    const float s = seen ? (s4[0] + s4[1]) + (s4[2] + s4[3]) : -INFINITY;
    const float m_new = fmaxf(m, wave_max(s));
    const float p = s == -INFINITY ? 0.f : expf(s - m_new);
    const float alpha = m == m_new ? 1.f : expf(m - m_new);
    l = l * alpha + wave_sum(p);
    m = m_new;
    ps[wave][lane] = p;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const f32x4 pv = *(const f32x4*)(&ps[wave][4 * (lane & 15)]);
    bool there[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) there[c] = vkey + c >= lo && vkey + c <= pos && v_held;
#pragma unroll
    for (int i = 0; i < H4; ++i) {
      float x = acc[i] * alpha;
#pragma unroll
      for (int c = 0; c < 4; ++c) x = fmaf(pv[c], there[c] ? v[i][c] : 0.f, x);
      acc[i] = x;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
#pragma unroll
  for (int i = 0; i < H4; ++i) {
    float x = acc[i];
    x += lane_dpp<TNX_DPP_XOR1>(x);
    x += lane_dpp<TNX_DPP_XOR2>(x);
    x += lane_dpp<TNX_DPP_HALF_MIRROR>(x);
    x += lane_dpp<TNX_DPP_MIRROR>(x);
    if ((lane & 15) == 0) os[wave][4 * i + (lane >> 4)] = x;
  }
  if (lane == 0) {
    ms[wave] = m;
    ls[wave] = l;
  }
  __syncthreads();
  for (int d = threadIdx.x; d < HD; d += 512) {
    float top = -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) top = fmaxf(top, ms[w]);
    float sum = 0.f, v = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float f = ms[w] == top ? 1.f : expf(ms[w] - top);       // (no wave is left out, as above)
      sum += f * ls[w];
      v += f * os[w][d];
    }
    a.out[at + d] = v * (1.f / sum);
  }
}

template <int HD>
int launch(const F32Attention& a, int num_tiles, int num_decode, hipStream_t stream) {
  if (num_tiles > 0) {
    constexpr int bytes = (4 * 32 * (HD + 4) + 256) * 4;
    static bool configured = false;
    if (!configured) {
      hipError_t e = hipFuncSetAttribute((const void*)attention_prompt_f32_kernel<HD>,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
      TNX_REQUIRE(e == hipSuccess, "attention_f32: cannot reserve %d bytes of LDS: %s", bytes, hipGetErrorString(e));
      configured = true;
    }
    const long long blocks = 4ll * num_tiles * a.num_heads;
    TNX_REQUIRE(blocks < (1ll << 31), "attention_f32: too many tiles");
    attention_prompt_f32_kernel<HD><<<(unsigned)blocks, 256, bytes, stream>>>(a);
    TNX_CHECK_LAUNCH("attention_prompt_f32");
  }
  if (num_decode > 0) {
    attention_decode_f32_kernel<HD><<<dim3(num_decode, a.num_heads), 512, 0, stream>>>(a);
    TNX_CHECK_LAUNCH("attention_decode_f32");
  }
  return 0;
}

}  // namespace

// `tile_run`, `tile_start`: the tiles of 128 queries of the runs of several tokens (`num_tiles` of them), `decode_runs`
// the runs of one token. `page_pad`: elements between the end of one page and the start of the next, a multiple of 8.
extern "C" int tnx_attention_f32(const float* q, const float* k_pages, const float* v_pages, const int* run_start,
                                 const int* cached_lens, const int* table, int table_width, int page_size, int num_pages,
                                 const int* tile_run, const int* tile_start, int num_tiles, int query_tile,
                                 const int* decode_runs, int num_decode, float* out, int num_heads, int num_kv,
                                 int head_size, int window, int page_pad, hipStream_t stream) {
  TNX_REQUIRE(num_heads > 0 && num_heads <= 65535 && num_kv > 0 && num_heads % num_kv == 0, "attention_f32: bad head counts");
  TNX_REQUIRE(page_pad >= 0 && page_pad % 8 == 0, "attention_f32: bad distance between pages");
  TNX_REQUIRE(page_size % 16 == 0 && page_size > 0, "attention_f32: page size %d is not a multiple of 16", page_size);
  TNX_REQUIRE(query_tile == 128, "attention_f32: tiles of 128 queries, got %d", query_tile);
  TNX_REQUIRE(num_tiles >= 0 && num_tiles < (1 << 28) && num_decode >= 0 && table_width > 0, "attention_f32: bad counts");
  TNX_REQUIRE(((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) % 16 == 0, "attention_f32: operands must be 16-byte aligned");
  F32Attention a;
  a.q = q; a.k_pages = k_pages; a.v_pages = v_pages; a.run_start = run_start; a.cached_lens = cached_lens;
  a.table = table; a.tile_run = tile_run; a.tile_start = tile_start; a.decode_runs = decode_runs; a.out = out;
  a.table_width = table_width; a.page_size = page_size; a.num_pages = num_pages; a.num_heads = num_heads;
  a.num_kv = num_kv; a.window = window; a.num_tiles = num_tiles;
  a.page_stride = (size_t)num_kv * page_size * head_size + page_pad;
  switch (head_size) {
    case 16: return launch<16>(a, num_tiles, num_decode, stream);
    case 32: return launch<32>(a, num_tiles, num_decode, stream);
    case 48: return launch<48>(a, num_tiles, num_decode, stream);
    case 64: return launch<64>(a, num_tiles, num_decode, stream);
    case 80: return launch<80>(a, num_tiles, num_decode, stream);
    case 96: return launch<96>(a, num_tiles, num_decode, stream);
    case 112: return launch<112>(a, num_tiles, num_decode, stream);
    case 128: return launch<128>(a, num_tiles, num_decode, stream);
    default: TNX_REQUIRE(false, "attention_f32: head size %d is not a multiple of 16 up to 128", head_size);
  }
}
