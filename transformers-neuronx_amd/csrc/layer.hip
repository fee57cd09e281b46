// Consecutive layers of a decode step of few rows in one launch: of each, queries, keys and values, attention over the cache, the
// output product, the two products of the feed-forward, and the norms and sums between them.
//
// What bounds such a step is the chain of its launches: five a layer of 4 to 6 us each, of which the bytes are one. Here the
// blocks of one launch stay and hand their results on through memory, five times a layer. A handoff is data and flag in one: the
// places are filled with a pattern that no result has (`NOT_YET`) before the launch, a producer stores its words past the caches, and
// a consumer asks for the words themselves until none of them is the pattern. Measured, us a handoff that all blocks make and all
// blocks wait for (1,024 words, 64 / 128 / 256 blocks): 1.1 / 1.5 / 2.0, and 2.8 beside a stream of 4 MB; with a flag a block beside the
// data 2.9 / - / 3.7, with one counter 2.8 / - / 4.9. Blocks beyond the ones that compute fetch what those read next into their XCD's L2
// (without them 18.4 us a layer for 16.8). us a layer, launches apart / so: bfloat16, 1,024 columns, 1 request of 100 tokens 23.1 / 16.9, 8 of
// 100 26.5 / 20.2, 1 of 1,500 27.7 / 20.2, 8 of 2,000 41.9 / 36.6; float32 3 of 70 34.4 / 26.8, 8 of 100 45.3 / 41.3, 4 of 1,000 54.2 / 36.0.
//
// A block waits only for blocks that run beside it: the layers are shared out among those that have joined (`join`), and who joins
// is on the chip and stays. A launch has a block that computes for every second compute unit (a unit has room for two of the bfloat16
// kernel's, 512 threads of 128 registers and 74 KB of LDS, and one of the float32 kernel's); where other launches leave no room for all of
// them (several engines on streams or in processes, units masked out), those that came do the work of all, and those that come later
// end at once. Blocks that fetch ahead wait for `AHEAD_TICKS` at most and then end as well. So whatever else runs, and however many
// such launches, every wait has its answer. It ends after `wait_most` questions all the same, some seconds: the block then goes on with
// results that are no numbers and says so in `failed`, which the host looks at where tokens reach it.
#include "common.h"

TNX_DEFINE_ERROR_API

namespace {

constexpr int NW = 8, THREADS = 64 * NW;      // waves of a block
constexpr int MOST_ROWS = 8;
constexpr int HD = 64;                        // the head size
constexpr int COLS = 8;                       // columns of a product's tile: its 8 waves share K
constexpr unsigned NOT_YET = 0xFFFFFFFFu;     // as a float, and as two bfloat16, no number, and none that a result is stored as
constexpr int CLOSED = 1 << 16;               // added to the number of blocks that asked to join, by who closes the launch to others
constexpr long long JOIN_TICKS = 1000, AHEAD_TICKS = 20000;     // of 10 ns

typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;

// What a layer has of its own.
struct LayerOf {
  const void *w_qkv, *w_out, *w_up, *w_down;          // bfloat16: tile order; float32: [columns][K]
  const float *b_qkv, *b_out, *b_up, *b_down;         // (zeros where there is none)
  const float *first_weight, *first_bias, *second_weight, *second_bias;     // the norms of what the two halves read (ones, zeros)
  void *k_pages, *v_pages;
};

// The places of a layer's handoffs, in words from the layer's first: queries, keys and values; the heads' results, and the parts
// of those whose keys are cut; the first sum, the feed-forward's inner values, the second sum.
struct Places {
  int qkv, mixed, parts, sum, inner, last, all;
};

constexpr int MOST_LAYERS = 30;               // (a launch's arguments are 4 KB at most)

struct Layers {
  const float* x;        // [rows][width] the stream, or, with `residual_normed`, what its norm reads
  float* out;            // [rows][width], float32
  const int *token_page, *token_off, *cached_lens, *table;
  unsigned* words;
  int* failed;
  Places at;
  float scale, eps;
  int rows, width, inner_width, act, center, residual_normed, first_normed;      // `first_normed` 0: the first layer's rows come as they are
  int table_width, page_shift, num_pages, page_pad, splits, chunk, layers, blocks;
  int join_most, wait_most;      // as many blocks at most join; questions of a wait
  LayerOf of[MOST_LAYERS];
};
static_assert(sizeof(Layers) <= 4096, "what a launch may take");

// A launch's arguments where they lie. `again`: from here on they are read again; what the compiler derives from them would else be
// kept from before the first layer in more scalar registers than there are.
typedef const __attribute__((address_space(4))) Layers* Args;
typedef const __attribute__((address_space(4))) LayerOf* ArgsOf;
template <typename P>
__device__ __forceinline__ P again(P p) {
  asm volatile("" : "+s"(p));
  return p;
}

// The thread's number, asked for where it is used: what the compiler derives from it (addresses above all) it then derives again in
// every phase of every layer, where it would keep hundreds of registers through all of them.
__device__ __forceinline__ int thread() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// ---- words that other blocks wrote

__device__ __forceinline__ void publish(unsigned* p, unsigned v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void publish(unsigned* p, unsigned v, unsigned next) {
  __hip_atomic_store((unsigned long long*)p, (unsigned long long)next << 32 | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Which of how many blocks this one is: the members of a launch, numbered from 0; -1: the launch goes on without it.
struct Member {
  int number, of;
};

// Asked by one thread. Two words behind those of the layers (-1 before the launch, as all of them): how many blocks have asked, and how
// many have joined where not all came. All have joined once as many have asked. Who has waited so long without another having come that
// going on with those there are would have lost no more (10 us a layer; a launch of 1 / n of the blocks takes n times as long) closes
// the launch to others and says how many there are by then: all of those are on the chip, and whoever asks later sees that it is closed.
__device__ __forceinline__ unsigned* gate_of(Args a) { return a->words + (size_t)a->layers * a->at.all; }
__device__ __forceinline__ unsigned ask_in(Args a, unsigned add) {
  return __hip_atomic_fetch_add(gate_of(a), add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
}
__device__ __forceinline__ Member join(Args a, unsigned number) {       // `number`: what `ask_in(a, 1)` said
  const unsigned most = a->join_most;
  if (number >= most) return {-1, 0};                    // (also where it is closed: `CLOSED` and more)
  unsigned came = number + 1;
  long long since = wall_clock64();
#pragma unroll 1
  for (;;) {
    const unsigned long long both = __hip_atomic_load((unsigned long long*)gate_of(a), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned asked = (unsigned)both + 1, joined = (unsigned)(both >> 32);
    const unsigned members = asked < CLOSED && asked >= most ? most : joined;
    // (all of them: numbered as blocks go to XCDs, for what was fetched ahead)
    if (members != NOT_YET) return {(int)members == a->blocks ? (int)blockIdx.x : (int)number, (int)members};
    if (asked >= CLOSED) continue;                       // (who closed it says so next)
    const long long now = wall_clock64();
    if (asked != came) {
      came = asked, since = now;
    } else if ((now - since) * came > JOIN_TICKS * a->layers * a->blocks) {
      const unsigned all = ask_in(a, CLOSED);
      if (all < CLOSED) __hip_atomic_store(gate_of(a) + 1, min(all, most), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_s_sleep(1);
  }
}

__device__ __forceinline__ unsigned float_word(float v) {
  const unsigned u = __float_as_uint(v);
  return u == NOT_YET ? 0x7FC00000u : u;
}
__device__ __forceinline__ unsigned pair_word(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  const bf16x2 two = {(bf16_t)a, (bf16_t)b};
  const unsigned u = __builtin_bit_cast(unsigned, two);
  return u == NOT_YET ? 0x7FC07FC0u : u;
}

// Reads past the caches of this unit and of its XCD (the scope of the device).
struct Shared {
  __amdgpu_buffer_rsrc_t base;
  __device__ __forceinline__ explicit Shared(const unsigned* p) : base(__builtin_amdgcn_make_buffer_rsrc((void*)p, 0, -1, 0x00020000)) {}
  __device__ __forceinline__ u32x4 four(int word) const {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(base, 4 * word, 0, 16));
  }
};

// Asks for N x 16 bytes (`word(i)`: the first of the four words of load i) until all are there, `most` times at most.
template <int N, typename Word>
__device__ __forceinline__ void await(const Shared& from, u32x4 (&v)[N], Word word, int most, bool& lost) {
#pragma unroll 1
  for (int asked = 0; asked < most; ++asked) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = from.four(word(i));
    bool there = true;
#pragma unroll
    for (int i = 0; i < N; ++i) there = there && v[i].x != NOT_YET && v[i].y != NOT_YET && v[i].z != NOT_YET && v[i].w != NOT_YET;
    if (__all(there) || lost) return;
  }
  lost = true;
}

// ---- a step's operand in LDS: [rows][K + PAD]

template <typename T>
struct Kind;
template <>
struct Kind<bf16_t> {
  // elements a word; loads of a job (8 columns x 128 of K) of a lane; keys of a tile of the attention
  static constexpr int PAD = 8, WORD = 2, LOADS = 2, KEYS = 64;
};
template <>
struct Kind<float> {
  static constexpr int PAD = 4, WORD = 1, LOADS = 4, KEYS = 32;
};

// Row `wave` of the rows: normed (or as it is) into LDS; its mean and 1 / deviation into `stat`. `PER` x 256 elements a lane's four.
template <typename T, int PER, typename Load>
__device__ __forceinline__ void norm_row(Args a, const float* weight, const float* bias, bool on, Load load, T* rows, int pitch, float (*stat)[2]) {
  const int tid = thread(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), width = a->width;
  if (wave >= a->rows) return;
  f32x4 gw[PER], gb[PER], v[PER];
  load(v, wave, lane);
  // (before the rows, these would be waited for before them)
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = min(256 * j + 4 * lane, width - 4);
    gw[j] = *(const f32x4*)(weight + i);
    gb[j] = *(const f32x4*)(bias + i);
  }
  float s = 0.f, q = 0.f;
#pragma unroll
  for (int j = 0; j < PER; ++j)
    if (256 * j + 4 * lane < width) s += (v[j].x + v[j].y) + (v[j].z + v[j].w);
  const float mean = on && a->center ? wave_sum(s) / (float)width : 0.f;
#pragma unroll
  for (int j = 0; j < PER; ++j)
    if (256 * j + 4 * lane < width) {
      const f32x4 d = v[j] - mean;
      q += (d.x * d.x + d.y * d.y) + (d.z * d.z + d.w * d.w);
    }
  const float rstd = on ? rsqrtf(wave_sum(q) / (float)width + a->eps) : 1.f;
  if (lane == 0) stat[wave][0] = mean, stat[wave][1] = rstd;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = 256 * j + 4 * lane;
    if (i >= width) continue;
    const f32x4 y = (v[j] - mean) * rstd * gw[j] + gb[j];       // (without a norm: itself)
    typedef T four __attribute__((ext_vector_type(4)));
    four o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (T)y[e];
    *(four*)(rows + wave * pitch + i) = o;
  }
}

// ---- products: tiles of 8 columns, K in steps of 128 that the waves take in turn

// Fragments of RT tiles x SC steps of the weight, asked for before the operand is there.
template <typename T, int SC, int RT>
struct Weights {
  u32x4 v[SC][RT][Kind<T>::LOADS];
  // steps 8 (chunk * SC + sc) + wave of tiles me.number + me.of (group * RT + j); what is beyond the end reads the last again (a load
  // that depended on anything would keep these registers from layer to layer)
  __device__ __forceinline__ void one(const T* w, int K, int tiles, Member me, int group, int chunk, int sc, int j) {
    const int tid = thread(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tile = min(me.number + me.of * (group * RT + j), tiles - 1), step = min(NW * (chunk * SC + sc) + wave, K / 128 - 1);
    if constexpr (sizeof(T) == 2) {
      // rows 0-7 of the matrix instruction's operand: the tile's columns over the first half of the step's K, rows 8-15 the
      // same columns over the second
      const int r = lane & 15, g = lane >> 4;
      const bf16_t* at = (const bf16_t*)w + (size_t)(tile >> 1) * 16 * K + (size_t)step * 2048 + (r >> 3) * 1024 + ((tile & 1) * 8 + (r & 7)) * 32 + 8 * g;
#pragma unroll
      for (int l = 0; l < 2; ++l) v[sc][j][l] = *(const u32x4*)(at + 512 * l);
    } else {
      const float* at = (const float*)w + (size_t)(tile * COLS + (lane & 7)) * K + step * 128 + 4 * (lane >> 3);
#pragma unroll
      for (int l = 0; l < 4; ++l) v[sc][j][l] = *(const u32x4*)(at + 32 * l);
    }
  }
  __device__ __forceinline__ void ask(const T* w, int K, int tiles, Member me, int group, int chunk) {
#pragma unroll
    for (int sc = 0; sc < SC; ++sc)
#pragma unroll
      for (int j = 0; j < RT; ++j) one(w, K, tiles, me, group, chunk, sc, j);
  }
};

// The sums of RT tiles: on the matrix unit, or a lane's share of one column and all rows. A wave leaves a tile's in LDS as [row][column].
template <typename T, int RT, int ROWS>
struct Sums;
template <int RT, int ROWS>
struct Sums<bf16_t, RT, ROWS> {
  f32x4 acc[RT];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int j = 0; j < RT; ++j) acc[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  template <int SC>
  __device__ __forceinline__ void add(const Weights<bf16_t, SC, RT>& w, int sc, const bf16_t* rows, int pitch, int k, int m_rows) {
    const int lane = thread() & 63, r = lane & 15, g = lane >> 4;
    const bf16_t* at = rows + min(r & 7, m_rows - 1) * pitch + k + 64 * (r >> 3) + 8 * g;
#pragma unroll
    for (int l = 0; l < 2; ++l) {
      const bf16x8 x = *(const bf16x8*)(at + 32 * l);
#pragma unroll
      for (int j = 0; j < RT; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w.v[sc][j][l]), x, acc[j], 0, 0, 0);
    }
  }
  // Element (row 4 (lane / 16) + i, column lane % 16) of the instruction's result counts where both are of the same half of K: those
  // of the second half, 40 lanes on, join those of the first.
  __device__ __forceinline__ void leave(float* red, int) {
    const int lane = thread() & 63;
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      f32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        unsigned lo, hi;
        swap_halves(__float_as_uint(lane_dpp<0x128>(acc[j][i])), lo, hi);       // (row_ror:8: lane ^ 8 of the 16)
        v[i] = acc[j][i] + __uint_as_float(hi);
      }
      if (lane < 32 && !(lane & 8)) *(f32x4*)(red + j * 64 + (lane & 7) * 8 + 4 * (lane >> 4)) = v;
    }
  }
};
template <int RT, int ROWS>
struct Sums<float, RT, ROWS> {
  f32x4 acc[RT][ROWS];      // (by element of the loads: short sums)
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int j = 0; j < RT; ++j)
#pragma unroll
      for (int m = 0; m < ROWS; ++m) acc[j][m] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  template <int SC>
  __device__ __forceinline__ void add(const Weights<float, SC, RT>& w, int sc, const float* rows, int pitch, int k, int m_rows) {
    const float* at = rows + k + 4 * ((thread() & 63) >> 3);
#pragma unroll
    for (int m = 0; m < ROWS; ++m) {
      if (m >= m_rows) break;
#pragma unroll
      for (int l = 0; l < 4; ++l) {
        const f32x4 x = *(const f32x4*)(at + m * pitch + 32 * l);
#pragma unroll
        for (int j = 0; j < RT; ++j) {
          const f32x4 v = __builtin_bit_cast(f32x4, w.v[sc][j][l]);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[j][m][e] = fmaf(v[e], x[e], acc[j][m][e]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);       // (else the operand of all rows is read before the first is used)
    }
  }
  __device__ __forceinline__ void leave(float* red, int m_rows) {
    const int lane = thread() & 63;
#pragma unroll
    for (int j = 0; j < RT; ++j)
#pragma unroll
      for (int m = 0; m < ROWS; ++m) {
        if (m >= m_rows) break;
        const float of_lane = (acc[j][m].x + acc[j][m].y) + (acc[j][m].z + acc[j][m].w), v = rows_sum(of_lane + lane_dpp<0x128>(of_lane));
        if (lane < 8) red[j * 64 + m * 8 + lane] = v;
      }
  }
};

// The block's tiles of one product. `stage(k0)`: the operand's elements of K from k0 on (`a->chunk` of them at most, or all) are in
// LDS for all when it returns; `early(mine, n, m)`: what the end adds, asked for before (`first`: of the first tiles, by the caller,
// before it waits for anything); `put(v0, v1, n, m, early)`: columns n, n + 1 of row m.
template <int RT, typename Early>
__device__ __forceinline__ auto of_first_tiles(Args a, Member me, int columns, Early early) {
  const int tid = thread(), tile = me.number + me.of * (tid >> 5), m = (tid >> 2) & 7;
  return early(tid < 32 * RT && tile < columns / COLS && m < a->rows, tile * COLS + 2 * (tid & 3), m);
}
template <typename T, int SC, int RT, int ROWS, typename First, typename Early, typename Stage, typename Put>
__device__ __forceinline__ void product(Args a, Member me, const T* w, int K, int columns, int chunk_k, Weights<T, SC, RT>& asked, const T* rows, int pitch,
                                        float* red, First first, Early early, Stage stage, Put put) {
  const int tid = thread(), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles = columns / COLS, steps = K / 128, turns = (steps + NW * SC - 1) / (NW * SC);
  typedef Sums<T, RT, ROWS> Made;
  if (me.number >= tiles) return;
  // the thread's two columns and row of the group's tiles: RT x 8 rows x 4 pairs
  const int j = tid >> 5, m = (tid >> 2) & 7, c = 2 * (tid & 3);
#pragma unroll 1
  for (int group = 0;; ++group) {
    const int tile = me.number + me.of * (group * RT + j), n = tile * COLS + c;
    const bool mine = tid < 32 * RT && tile < tiles && m < a->rows;
    const First extra = group == 0 ? first : early(mine, n, m);
    Made sums;
    sums.clear();
    const bool more = me.number + me.of * (group + 1) * RT < tiles;
#pragma unroll 1
    for (int k0 = 0; k0 < K; k0 += chunk_k) {
      if (group == 0 || chunk_k < K) stage(k0);
      const int from = k0 / (128 * NW * SC), last = min(turns, (k0 + chunk_k + 128 * NW * SC - 1) / (128 * NW * SC));
#pragma unroll 1
      for (int turn = from; turn < last; ++turn) {
#pragma unroll
        for (int sc = 0; sc < SC; ++sc) {
          const int step = NW * (turn * SC + sc) + wave;
          if (step < steps) sums.add(asked, sc, rows, pitch, step * 128 - k0, a->rows);
        }
        if (turn + 1 < turns) asked.ask(w, K, tiles, me, group, turn + 1);
        else if (more) asked.ask(w, K, tiles, me, group + 1, 0);
      }
    }
    sums.leave(red + wave * RT * 64, a->rows);
    __syncthreads();
    if (mine) {
      f32x2 v[NW];
#pragma unroll
      for (int i = 0; i < NW; ++i) v[i] = *(const f32x2*)(red + (i * RT + j) * 64 + m * 8 + c);
      v[0] = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
      put(v[0].x, v[0].y, n, m, extra);
    }
    if (!more) return;
    __syncthreads();
  }
}

// Words of `count` x 16 bytes a row into LDS, as they came.
template <typename T>
__device__ __forceinline__ void stage_words(const unsigned* from, int words_row, int word0, int words, int m_rows, T* rows, int pitch, int most,
                                            bool& lost) {
  const Shared src(from);
  const int per_row = words / 4, all = per_row * m_rows;
  const int tid = thread();
#pragma unroll 1
  for (int at = tid; at - tid < all; at += 2 * THREADS) {
    int row[2], four[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int q = min(at + i * THREADS, all - 1);
      row[i] = q / per_row, four[i] = q - row[i] * per_row;
    }
    u32x4 v[2];
    await<2>(src, v, [&](int i) { return row[i] * words_row + word0 + 4 * four[i]; }, most, lost);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (at + i * THREADS < all) *(u32x4*)((char*)(rows + row[i] * pitch) + 16 * four[i]) = v[i];
  }
}

// ---- attention

// How the keys of a request (`held` in the cache, 64 a tile) are cut: up to a tile a wave of one block not at all, beyond that into
// shares of four tiles or more (us a layer, bfloat16 of 1,024: 1 request of 1,500 by shares of 4, 8 and 16 tiles 20.2, 22.4, 25.1; 4 of
// 600 22.0, 23.5, 22.4; but 2 of 300 of 512 columns, 5 tiles, 19.1 cut and 17.2 whole).
__device__ __forceinline__ int tiles_per_share(int held, int splits) {
  const int tiles = (held + 63) / 64;
  return tiles <= NW ? NW : max(4, (tiles + splits - 1) / splits);
}
__device__ __forceinline__ int shares_of(int held, int splits) {
  const int tiles = (held + 63) / 64, per = tiles_per_share(held, splits);
  return max(1, (tiles + per - 1) / per);
}

// A (row, head, share of its keys) as a block attends to it: looked up once, for all layers.
struct Item {
  int row, h, share, held, page;      // `page`: of this wave's first tile
};
template <int KEYS>      // of a tile
__device__ __forceinline__ Item item_of(Args a, int item) {
  const int heads = a->width / HD, pairs = a->rows * heads, wave = __builtin_amdgcn_readfirstlane(thread() >> 6);
  Item i;
  i.share = item / pairs;
  const int at = item - i.share * pairs;
  i.row = at / heads, i.h = at - i.row * heads;
  i.held = a->cached_lens[i.row];
  if (i.share >= shares_of(i.held, a->splits)) i.share = -1;
  const int key0 = min(64 * max(i.share, 0) * tiles_per_share(i.held, a->splits) + KEYS * wave, max(i.held - 1, 0));
  i.page = min(max(a->table[(size_t)i.row * a->table_width + (key0 >> a->page_shift)], 0), a->num_pages - 1);
  return i;
}

struct __attribute__((aligned(16))) Softmax {
  float o[NW][HD];
  float own[2 * HD];        // float32: the row's own key and value
  float m[NW], l[NW];
};

constexpr int PART = HD + 4;      // words of a share's partial result: its sums, its maximum, its sum of weights, two unused

// One row's head and share of its keys, bfloat16: keys and values of 64 on the matrix unit, as `attention_decode_mfma` has them
// (attention.hip): the query is all 16 columns of S^T = K q, row r of key block kb is key 32 (kb / 2) + 8 (r / 4) + 4 (kb % 2) + r % 4.
__device__ __forceinline__ void attend(Args a, ArgsOf of, const unsigned* words, const Item& item, Softmax& sm, bool& lost, bf16_t) {
  const int tid = thread(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
  const int row = item.row, h = item.h, share = item.share, held = item.held, heads = a->width / HD, page_size = 1 << a->page_shift;
  const int tiles = (held + 63) / 64, per = tiles_per_share(held, a->splits);
  const int end = min(tiles, (share + 1) * per);
  const int* tab = a->table + (size_t)row * a->table_width;
  const size_t head_stride = (size_t)page_size * HD, page_stride = (size_t)heads * head_stride + a->page_pad;
  bf16x8 kf[4][2], vf[4][2];
  auto page_of = [&](int t) { return min(max(tab[__builtin_amdgcn_readfirstlane(64 * t) >> a->page_shift], 0), a->num_pages - 1); };
  auto load = [&](int t, int page) {
    const int key0 = __builtin_amdgcn_readfirstlane(64 * t);
    const bf16_t* kp = (const bf16_t*)of->k_pages + (size_t)page * page_stride + (size_t)h * head_stride + (size_t)(key0 & (page_size - 1)) * HD;
    const bf16_t* vp = (const bf16_t*)of->v_pages + (size_t)page * page_stride + (size_t)h * head_stride + (key0 & (page_size - 1));
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        kf[kb][ks] = *(const bf16x8*)(kp + (32 * (kb >> 1) + 8 * (r >> 2) + 4 * (kb & 1) + (r & 3)) * HD + 32 * ks + 8 * g);
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int db = 0; db < 4; ++db) vf[db][st] = *(const bf16x8*)(vp + (size_t)(16 * db + r) * page_size + 32 * st + 8 * g);
  };
  int t = share * per + wave;
  if (t < end) load(t, item.page);
  const Shared mine(words + a->at.qkv + (size_t)row * (3 * a->width / 2));
  u32x4 qw[2];
  await<2>(mine, qw, [&](int ks) { return h * (HD / 2) + 16 * ks + 4 * g; }, a->wait_most, lost);
  bf16x8 qf[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) qf[ks] = __builtin_bit_cast(bf16x8, qw[ks]);
  float m = -INFINITY, l = 0.f;
  f32x4 o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) o[db] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (; t < end; t += NW) {
    f32x4 sc[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      sc[kb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) sc[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kb][ks], qf[ks], sc[kb], 0, 0, 0);
    }
    const bool edge = 64 * t + 64 > held;
    float mx = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (edge && 64 * t + 32 * (kb >> 1) + 8 * g + 4 * (kb & 1) + i >= held) sc[kb][i] = -INFINITY;
        mx = fmaxf(mx, sc[kb][i]);
      }
    const float m_new = fmaxf(m, rows_max(mx)), m_safe = m_new == -INFINITY ? 0.f : m_new, alpha = __expf(m - m_safe);
    float sum = 0.f;
    bf16x8 pf[2];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = __expf(sc[kb][i] - m_safe);
        sum += p;
        pf[kb >> 1][4 * (kb & 1) + i] = (bf16_t)p;
      }
    l = l * alpha + sum;
    m = m_new;
    if (edge) {
      // what lies beyond the request's keys may be anything: its weights are zero, and it must be a number
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (64 * t + 32 * st + 8 * g + e >= held) {
#pragma unroll
            for (int db = 0; db < 4; ++db) vf[db][st][e] = 0;
          }
    }
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      o[db] *= alpha;
#pragma unroll
      for (int st = 0; st < 2; ++st) o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[db][st], pf[st], o[db], 0, 0, 0);
    }
    if (t + NW < end) load(t + NW, page_of(t + NW));
  }
  l = rows_sum(l);
  if (share == 0 && wave == NW - 1) {
    // the row's own key and value, which this launch has made
    u32x4 kv[6];
    await<6>(mine, kv, [&](int i) {
      return i < 2 ? a->width / 2 + h * (HD / 2) + 16 * i + 4 * g : a->width + h * (HD / 2) + 8 * (i - 2) + 4 * (g >> 1);
    }, a->wait_most, lost);
    float s = 0.f;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const bf16x8 key = __builtin_bit_cast(bf16x8, kv[ks]);
#pragma unroll
      for (int e = 0; e < 8; ++e) s = fmaf((float)qf[ks][e], (float)key[e], s);
    }
    s = rows_sum(s);
    const float m_new = fmaxf(m, s), m_safe = m_new == -INFINITY ? 0.f : m_new, alpha = __expf(m - m_safe), p = __expf(s - m_safe);
    const float pr = (float)(bf16_t)p;          // (as the weights of the other keys)
    l = l * alpha + p;
    m = m_new;
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      const bf16x8 vv = __builtin_bit_cast(bf16x8, kv[2 + db]);       // elements 16 db + 8 (g / 2) + 0..7 of the head
#pragma unroll
      for (int i = 0; i < 4; ++i) o[db][i] = fmaf(pr, (float)((g & 1) ? vv[4 + i] : vv[i]), o[db][i] * alpha);
    }
  }
  if (r == 0) {
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) sm.o[wave][16 * db + 4 * g + i] = o[db][i];
  }
  if (lane == 0) sm.m[wave] = m, sm.l[wave] = l;
}

// The same in float32: 32 keys a turn. For the scores two lanes take a key and a half of the head each; for the weighted values
// eight lanes take the 32 keys of an element, four each.
__device__ __forceinline__ void attend(Args a, ArgsOf of, const unsigned* words, const Item& item, Softmax& sm, bool& lost, float) {
  const int tid = thread(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = item.row, h = item.h, share = item.share, held = item.held, heads = a->width / HD, page_size = 1 << a->page_shift;
  const int tiles = (held + 63) / 64, per = tiles_per_share(held, a->splits);
  const int end = 2 * min(tiles, (share + 1) * per);
  const int* tab = a->table + (size_t)row * a->table_width;
  const size_t head_stride = (size_t)page_size * HD, page_stride = (size_t)heads * head_stride + a->page_pad;
  f32x4 kk[8], vv[8];
  const int key_of = lane & 31, half = lane >> 5, group = lane & 7, first_d = lane >> 3;
  auto page_of = [&](int t) { return min(max(tab[__builtin_amdgcn_readfirstlane(32 * t) >> a->page_shift], 0), a->num_pages - 1); };
  auto load = [&](int t, int page) {
    const int key0 = __builtin_amdgcn_readfirstlane(32 * t);
    const float* kp = (const float*)of->k_pages + (size_t)page * page_stride + (size_t)h * head_stride +
                      (size_t)((key0 & (page_size - 1)) + key_of) * HD + 32 * half;
    const float* vp = (const float*)of->v_pages + (size_t)page * page_stride + (size_t)h * head_stride + (key0 & (page_size - 1)) + 4 * group;
#pragma unroll
    for (int i = 0; i < 8; ++i) kk[i] = *(const f32x4*)(kp + 4 * i);
#pragma unroll
    for (int i = 0; i < 8; ++i) vv[i] = *(const f32x4*)(vp + (size_t)(first_d + 8 * i) * page_size);
  };
  int t = 2 * share * per + wave;
  if (t < end) load(t, item.page);
  const Shared mine(words + a->at.qkv + (size_t)row * (3 * a->width));
  // the query, and the row's own key and value, which this launch has made, come together and wait in LDS, the query where the wave's
  // result will lie
  f32x4* const qs = (f32x4*)sm.o[wave];
  const bool own = share == 0 && wave == NW - 1;
  {
    u32x4 got[1];
    const int which = min(lane >> 4, 2);
    await<1>(mine, got, [&](int) { return which * a->width + h * HD + 4 * (lane & 15); }, a->wait_most, lost);
    if (lane < 16) qs[lane] = __builtin_bit_cast(f32x4, got[0]);
    else if (own && lane < 48) ((f32x4*)sm.own)[lane - 16] = __builtin_bit_cast(f32x4, got[0]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  float m = -INFINITY, l = 0.f, o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = 0.f;
#pragma unroll 1
  for (; t < end; t += NW) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const f32x4 q = qs[8 * half + i];
#pragma unroll
      for (int e = 0; e < 4; ++e) s = fmaf(q[e], kk[i][e], s);
    }
    unsigned lo, hi;
    swap_halves(__float_as_uint(s), lo, hi);
    s = 32 * t + key_of < held ? __uint_as_float(lo) + __uint_as_float(hi) : -INFINITY;
    const float m_new = fmaxf(m, wave_max(s));
    const float p = s == -INFINITY ? 0.f : expf(s - m_new), alpha = m == m_new ? 1.f : expf(m - m_new);
    l = l * alpha + 0.5f * wave_sum(p);          // (a key's weight lies with two lanes)
    m = m_new;
    float pv[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) pv[e] = __shfl(p, 4 * group + e);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float x = o[i] * alpha;
#pragma unroll
      for (int e = 0; e < 4; ++e) x = fmaf(pv[e], 32 * t + 4 * group + e < held ? vv[i][e] : 0.f, x);
      o[i] = x;
    }
    if (t + NW < end) load(t + NW, page_of(t + NW));
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float x = o[i];
    x += lane_dpp<TNX_DPP_XOR1>(x);
    x += lane_dpp<TNX_DPP_XOR2>(x);
    x += lane_dpp<TNX_DPP_HALF_MIRROR>(x);
    o[i] = x;
  }
  if (own) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const f32x4 q = qs[8 * half + i], key = ((f32x4*)sm.own)[8 * half + i];
#pragma unroll
      for (int e = 0; e < 4; ++e) s = fmaf(q[e], key[e], s);
    }
    unsigned lo, hi;
    swap_halves(__float_as_uint(s), lo, hi);
    s = __uint_as_float(lo) + __uint_as_float(hi);
    const float m_new = fmaxf(m, s), p = expf(s - m_new), alpha = m == m_new ? 1.f : expf(m - m_new);
    l = l * alpha + p;
    m = m_new;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = fmaf(p, sm.own[HD + first_d + 8 * i], o[i] * alpha);
  }
  if (group == 0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) sm.o[wave][first_d + 8 * i] = o[i];
  }
  if (lane == 0) sm.m[wave] = m, sm.l[wave] = l;
}

// What exponentials the two kinds take, as their own kernels do.
__device__ __forceinline__ float weight_of(float d, bf16_t) { return __expf(d); }
__device__ __forceinline__ float weight_of(float d, float) { return expf(d); }

// The waves' results of a (row, head, share) joined and handed on: the head's result, or, where any row's keys are cut, the share's part.
template <typename T>
__device__ __forceinline__ void join_waves(Args a, unsigned* words, const Item& item, bool cut, const Softmax& sm) {
  const int d = thread();
  if (d >= HD) return;
  const int row = item.row, h = item.h, share = item.share, heads = a->width / HD;
  float top = sm.m[0];
#pragma unroll
  for (int w = 1; w < NW; ++w) top = fmaxf(top, sm.m[w]);
  const float safe = top == -INFINITY ? 0.f : top;
  float sum = 0.f, v = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float f = weight_of(sm.m[w] - safe, T());
    sum += sm.l[w] * f;
    v += sm.o[w][d] * f;
  }
  if (!cut) {
    const float out = v / sum;
    if constexpr (sizeof(T) == 2) {
      const float next = lane_dpp<TNX_DPP_XOR1>(out);
      if (!(d & 1)) publish(words + a->at.mixed + (size_t)row * (a->width / 2) + h * (HD / 2) + d / 2, pair_word(out, next));
    } else {
      publish(words + a->at.mixed + (size_t)row * a->width + h * HD + d, float_word(out));
    }
  } else {
    unsigned* p = words + a->at.parts + (size_t)((row * heads + h) * a->splits + share) * PART;
    publish(p + d, float_word(v));
    if (d < 4) publish(p + HD + d, d == 0 ? float_word(top) : d == 1 ? float_word(sum) : 0u);
  }
}

// The rows' heads from the parts of their shares (at most N), into LDS.
template <typename T, int N>
__device__ __forceinline__ void stage_parts(Args a, const unsigned* words, T* rows, int pitch, bool& lost) {
  const int heads = a->width / HD, all = a->rows * heads * (HD / 4);
  const Shared src(words + a->at.parts);
  const int tid = thread();
#pragma unroll 1
  for (int at = tid; at - tid < all; at += THREADS) {
    const int q = min(at, all - 1), pair = q / (HD / 4), d = 4 * (q % (HD / 4)), row = pair / heads;
    const int shares = shares_of(a->cached_lens[row], a->splits);
    u32x4 got[2 * N];
    await<2 * N>(src, got, [&](int i) { return (pair * a->splits + min(i >> 1, shares - 1)) * PART + ((i & 1) ? d : HD); }, a->wait_most, lost);
    float top = -INFINITY;
#pragma unroll
    for (int s = 0; s < N; ++s) top = fmaxf(top, __uint_as_float(got[2 * s].x));
    const float safe = top == -INFINITY ? 0.f : top;
    float sum = 0.f;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < N; ++s) {
      if (s >= shares) continue;
      const float f = weight_of(__uint_as_float(got[2 * s].x) - safe, T());
      sum += f * __uint_as_float(got[2 * s].y);
      v += f * __builtin_bit_cast(f32x4, got[2 * s + 1]);
    }
    typedef T four __attribute__((ext_vector_type(4)));
    four out;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = (T)(v[e] / sum);
    if (at < all) *(four*)(rows + row * pitch + (pair - row * heads) * HD + d) = out;
  }
}

// ---- weights that come into an XCD's L2 before its blocks ask for them

// The tiles that the blocks of this one's XCD take of a matrix (every eighth: blocks go to XCDs in turn), one word of every 128 bytes.
template <typename T>
__device__ __forceinline__ void touch(const void* w, int K, int columns, int first, int waves) {
  const int tid = thread(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), xcd = blockIdx.x & 7;
  const int lines = K * COLS * (int)sizeof(T) / 128, parts = (lines + 255) / 256, tiles = columns / COLS;
  const int mine = (tiles - xcd + 7) / 8;
#pragma unroll 1
  for (int job = first + wave; job < mine * parts; job += waves) {
    const int tile = xcd + 8 * (job / parts), line0 = (job % parts) * 256 + lane;
    unsigned v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int line = min(line0 + 64 * i, lines - 1);
      size_t at;
      if constexpr (sizeof(T) == 2) at = (size_t)(tile >> 1) * 32 * K + (size_t)(line >> 2) * 1024 + (tile & 1) * 512 + (line & 3) * 128;
      else at = (size_t)tile * COLS * K * 4 + (size_t)line * 128;
      v[i] = *(const unsigned*)((const char*)w + at);
    }
    asm volatile("" ::"v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]));
  }
}

// The vectors of a layer, one of eight a wave of the first block of helpers; and the first keys and values of every share of a
// head's that a block of this XCD takes.
__device__ __forceinline__ void touch_vectors(Args a, ArgsOf of, int first) {
  const int tid = thread(), wave = __builtin_amdgcn_readfirstlane(tid >> 6), W = a->width;
  if (first != 0) return;
  const float* v = wave == 0 ? of->first_weight : wave == 1 ? of->first_bias : wave == 2 ? of->b_qkv : wave == 3 ? of->b_out :
                   wave == 4 ? of->second_weight : wave == 5 ? of->second_bias : wave == 6 ? of->b_up : of->b_down;
  const int n = wave == 2 ? 3 * W : wave == 6 ? a->inner_width : W;
  float x[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) x[i] = v[min((64 * i + (tid & 63)) * 32, n - 1)];
  asm volatile("" ::"v"(x[0]), "v"(x[1]));
}
template <typename T>
__device__ __forceinline__ void touch_cache(Args a, ArgsOf of, int first, int waves) {
  const int tid = thread(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int heads = a->width / HD, pairs = a->rows * heads, items = pairs * a->splits, page_size = 1 << a->page_shift;
  const size_t head_stride = (size_t)page_size * HD, page_stride = (size_t)heads * head_stride + a->page_pad;
#pragma unroll 1
  for (int job = first + wave; job < (items + 7) / 8 * NW; job += waves) {
    const int item = (job / NW) * 8 + (blockIdx.x & 7), share = item / pairs, row = (item - share * pairs) / heads, h = item - share * pairs - row * heads;
    if (item >= items) continue;
    const int held = a->cached_lens[row], per = tiles_per_share(held, a->splits), t = share * per + job % NW;
    if (t >= min((held + 63) / 64, (share + 1) * per)) continue;
    const int key0 = 64 * t, page = min(max(a->table[(size_t)row * a->table_width + (key0 >> a->page_shift)], 0), a->num_pages - 1);
    const size_t head = (size_t)page * page_stride + (size_t)h * head_stride;
    const T* kp = (const T*)of->k_pages + head + (size_t)((key0 & (page_size - 1)) + lane) * HD;
    const T* vp = (const T*)of->v_pages + head + (size_t)lane * page_size + (key0 & (page_size - 1));
    const unsigned k = *(const unsigned*)kp, v = *(const unsigned*)vp;
    asm volatile("" ::"v"(k), "v"(v));
    if constexpr (sizeof(T) == 4) {
      const unsigned k2 = *(const unsigned*)(kp + 32), v2 = *(const unsigned*)(vp + 32);
      asm volatile("" ::"v"(k2), "v"(v2));
    }
  }
}

// Whether a word came in time.
__device__ __forceinline__ bool until(const unsigned* p) {
  const long long since = wall_clock64();
  while (__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == NOT_YET) {
    if (wall_clock64() - since > AHEAD_TICKS) return false;
    __builtin_amdgcn_s_sleep(4);
  }
  return true;
}

// The blocks beyond the first `blocks` run ahead of those: a matrix is fetched when what is multiplied two matrices before it is there.
// What they fetch is a hint and the place that one holds is another block's: where the layers do not come on for 0.2 ms (the keys of 8
// requests of 2,000 tokens in float32 take a quarter of that), they end.
template <typename T>
__device__ void run_ahead(Args a) {
  const int helpers = (gridDim.x - a->blocks) / 8, first = (blockIdx.x - a->blocks) / 8 * NW, waves = helpers * NW;
#pragma unroll 1
  for (int l = 0; l < a->layers; ++l) {
    ArgsOf of = &a->of[l];
    const unsigned *words = a->words + (size_t)l * a->at.all, *before = words - a->at.all;
    if (l > 0 && !until(before + a->at.sum)) return;
    touch<T>(of->w_qkv, a->width, 3 * a->width, first, waves);
    touch_vectors(a, of, first);
    touch_cache<T>(a, of, first, waves);
    if (l > 0 && !until(before + a->at.inner)) return;
    touch<T>(of->w_out, a->width, a->width, first, waves);
    if (l > 0 && !until(before + a->at.last)) return;
    touch<T>(of->w_up, a->width, a->inner_width, first, waves);
    if (l > 0 && !until(words + a->at.qkv)) return;
    touch<T>(of->w_down, a->inner_width, a->width, first, waves);
  }
}

// bytes of LDS in which the waves' sums meet
template <typename T, int RT>
constexpr int red_bytes() { return NW * RT * 64 * 4; }

// One block's part of the layers, phase by phase: what a phase needs it derives from the arguments again.
// Widths of up to 1,024, a step of 128 a wave. SCD: steps of the inner width that a wave takes at a time; RQ, RU: tiles of a block that
// are made together of queries, keys and values, and of the feed-forward's first product; ROWS: as many as the sums have room for.
template <typename T, int ROWS, int SCD, int RQ, int RU>
struct Block {
  static constexpr int PER = 4, PAD = Kind<T>::PAD, WORD = Kind<T>::WORD, KEYS = Kind<T>::KEYS;
  struct Two { f32x2 bias, onto, weight, shift; };      // what the end adds to two columns: bias, residual, and the norm of the latter
  struct Place { f32x2 bias; int page, off; };
  char* smem;
  float (*stat1)[2];
  float (*stat2)[2];
  Softmax* sm;
  Member me;
  Item mine;
  bool cut;              // some row's keys are cut into shares
  bool lost;

  __device__ __forceinline__ float* red() const { return (float*)smem; }
  __device__ __forceinline__ T* rows() const { return (T*)(smem + red_bytes<T, (RQ > RU ? RQ : RU)>()); }
  __device__ __forceinline__ T* down_rows() const { return (T*)(smem + red_bytes<T, 1>()); }
  static __device__ __forceinline__ unsigned* words_of(Args a, int layer) { return a->words + (size_t)layer * a->at.all; }
  // the sum that the layer before left
  static __device__ __forceinline__ const unsigned* before(Args a, int layer) { return words_of(a, layer - 1) + a->at.last; }
  // two words of a row that was there when it was normed
  static __device__ __forceinline__ f32x2 two_words(const unsigned* p) {
    const unsigned long long w = __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return (f32x2){__uint_as_float((unsigned)w), __uint_as_float((unsigned)(w >> 32))};
  }
  static __device__ __forceinline__ f32x2 with_residual(Args a, float v0, float v1, const Two& t, const float (*stat)[2], int m) {
    f32x2 r = t.onto;
    if (a->residual_normed) r = (r - stat[m][0]) * stat[m][1] * t.weight + t.shift;
    return (f32x2){v0, v1} + t.bias + r;
  }
  static __device__ __forceinline__ void publish_two(unsigned* to, float v0, float v1) {
    publish(to, float_word(v0), float_word(v1));
  }
  // two columns of an operand of the next product
  static __device__ __forceinline__ void publish_operand(unsigned* to, int at, float v0, float v1) {
    if constexpr (sizeof(T) == 2) publish(to + at / 2, pair_word(v0, v1));
    else publish_two(to + at, v0, v1);
  }
  // a row's words as they come, for `norm_row`
  __device__ __forceinline__ void row_words(Args a, const unsigned* from, f32x4 (&v)[PER], int wave, int lane) {
    const Shared src(from + (size_t)wave * a->width);
    u32x4 got[PER];
    await<PER>(src, got, [&](int j) { return min(256 * j + 4 * lane, a->width - 4); }, a->wait_most, lost);
#pragma unroll
    for (int j = 0; j < PER; ++j) v[j] = __builtin_bit_cast(f32x4, got[j]);
  }

  // queries, keys and values
  __device__ __forceinline__ void project(Args args, int at_layer) {
    Args a = again(args);
    const int layer = again(at_layer), W = a->width;
    ArgsOf of = &a->of[layer];
    const bool normed = layer > 0 || a->first_normed;
    Weights<T, 1, RQ> asked;
    asked.ask((const T*)of->w_qkv, W, 3 * W / COLS, me, 0, 0);
    auto early = [&](bool mine, int n, int m) {
      Place p{{0.f, 0.f}, -1, 0};
      if (mine) p.bias = *(const f32x2*)(of->b_qkv + n), p.page = a->token_page[m], p.off = a->token_off[m];
      return p;
    };
    const Place first = of_first_tiles<RQ>(a, me, 3 * W, early);
    norm_row<T, PER>(a, of->first_weight, of->first_bias, normed, [&](f32x4 (&v)[PER], int wave, int lane) {
      if (layer == 0) {
#pragma unroll
        for (int j = 0; j < PER; ++j) v[j] = *(const f32x4*)(a->x + (size_t)wave * W + min(256 * j + 4 * lane, W - 4));
      } else {
        row_words(a, before(a, layer), v, wave, lane);
      }
    }, rows(), W + PAD, stat1);
    __syncthreads();
    product<T, 1, RQ, ROWS>(a, me, (const T*)of->w_qkv, W, 3 * W, W, asked, rows(), W + PAD, red(), first, early,
      [](int) {},
      [&](float v0, float v1, int n, int m, const Place& p) {
        v0 += p.bias.x, v1 += p.bias.y;
        if (n < W) v0 *= a->scale, v1 *= a->scale;
        publish_operand(words_of(a, layer) + a->at.qkv, m * 3 * W + n, v0, v1);
        if (n < W || p.page < 0 || p.page >= a->num_pages) return;
        const int page_size = 1 << a->page_shift, in = n >= 2 * W ? n - 2 * W : n - W, h = in / HD, d = in % HD;
        const size_t head = (size_t)p.page * ((size_t)(W / HD) * page_size * HD + a->page_pad) + (size_t)h * page_size * HD;
        if (n < 2 * W) {
          T* k = (T*)of->k_pages + head + (size_t)p.off * HD + d;
          k[0] = (T)v0, k[1] = (T)v1;
        } else {
          T* v = (T*)of->v_pages + head + (size_t)d * page_size + p.off;
          v[0] = (T)v0, v[page_size] = (T)v1;
        }
      });
  }

  // attention: a (row, head, share of its keys) a block, `mine` the first
  __device__ __forceinline__ void mix(Args a, int layer) {
    const int items = a->rows * (a->width / HD) * a->splits;
#pragma unroll 1
    for (int at = me.number; at < items; at += me.of) {
      if (at != me.number) mine = item_of<KEYS>(a, at);
      if (mine.share < 0) continue;
      attend(a, &a->of[layer], words_of(a, layer), mine, *sm, lost, T());
      __syncthreads();
      join_waves<T>(a, words_of(a, layer), mine, cut, *sm);
      __syncthreads();
    }
    if (items > me.of) mine = item_of<KEYS>(a, min(me.number, items - 1));
  }

  // attention, the output product and the first sum (whose weights are asked for before a block attends)
  __device__ __forceinline__ void put_out(Args args, int at_layer) {
    Args a = again(args);
    const int layer = again(at_layer), W = a->width;
    ArgsOf of = &a->of[layer];
    Weights<T, 1, 1> asked;
    asked.ask((const T*)of->w_out, W, W / COLS, me, 0, 0);
    auto early = [&](bool mine, int n, int m) {
      Two t{};
      if (mine) {
        t.bias = *(const f32x2*)(of->b_out + n);
        t.onto = layer ? two_words(before(a, layer) + m * W + n) : *(const f32x2*)(a->x + (size_t)m * W + n);
        if (a->residual_normed) t.weight = *(const f32x2*)(of->first_weight + n), t.shift = *(const f32x2*)(of->first_bias + n);
      }
      return t;
    };
    const Two first = of_first_tiles<1>(a, me, W, early);
    mix(a, layer);
    product<T, 1, 1, ROWS>(a, me, (const T*)of->w_out, W, W, W, asked, rows(), W + PAD, red(), first, early,
      [&](int) {
        if (!cut) stage_words<T>(words_of(a, layer) + a->at.mixed, W / WORD, 0, W / WORD, a->rows, rows(), W + PAD, a->wait_most, lost);
        else if (a->splits <= 2) stage_parts<T, 2>(a, words_of(a, layer), rows(), W + PAD, lost);
        else stage_parts<T, 8>(a, words_of(a, layer), rows(), W + PAD, lost);
        __syncthreads();
      },
      [&](float v0, float v1, int n, int m, const Two& t) {
        const f32x2 v = with_residual(a, v0, v1, t, stat1, m);
        publish_two(words_of(a, layer) + a->at.sum + m * W + n, v.x, v.y);
      });
  }

  // the feed-forward's first product
  __device__ __forceinline__ void go_up(Args args, int at_layer) {
    Args a = again(args);
    const int layer = again(at_layer), W = a->width, F = a->inner_width;
    ArgsOf of = &a->of[layer];
    Weights<T, 1, RU> asked;
    asked.ask((const T*)of->w_up, W, F / COLS, me, 0, 0);
    auto early = [&](bool mine, int n, int) {
      return mine ? *(const f32x2*)(of->b_up + n) : (f32x2){0.f, 0.f};
    };
    const f32x2 first = of_first_tiles<RU>(a, me, F, early);
    __syncthreads();             // (the operand before is read)
    norm_row<T, PER>(a, of->second_weight, of->second_bias, true, [&](f32x4 (&v)[PER], int wave, int lane) {
      row_words(a, words_of(a, layer) + a->at.sum, v, wave, lane);
    }, rows(), W + PAD, stat2);
    __syncthreads();
    product<T, 1, RU, ROWS>(a, me, (const T*)of->w_up, W, F, W, asked, rows(), W + PAD, red(), first, early,
      [](int) {},
      [&](float v0, float v1, int n, int m, f32x2 bias) {
        publish_operand(words_of(a, layer) + a->at.inner, m * F + n, apply_act(v0 + bias.x, a->act), apply_act(v1 + bias.y, a->act));
      });
  }

  // its second, and the second sum
  __device__ __forceinline__ void go_down(Args args, int at_layer) {
    Args a = again(args);
    const int layer = again(at_layer), W = a->width, F = a->inner_width;
    ArgsOf of = &a->of[layer];
    Weights<T, SCD, 1> asked;
    asked.ask((const T*)of->w_down, F, W / COLS, me, 0, 0);
    const int pitch = min(a->chunk, F) + PAD;
    auto early = [&](bool mine, int n, int m) {
      Two t{};
      if (mine) {
        t.bias = *(const f32x2*)(of->b_down + n);
        t.onto = two_words(words_of(a, layer) + a->at.sum + m * W + n);
        if (a->residual_normed) t.weight = *(const f32x2*)(of->second_weight + n), t.shift = *(const f32x2*)(of->second_bias + n);
      }
      return t;
    };
    const Two first = of_first_tiles<1>(a, me, W, early);
    product<T, SCD, 1, ROWS>(a, me, (const T*)of->w_down, F, W, a->chunk, asked, down_rows(), pitch, red(), first, early,
      [&](int k0) {
        __syncthreads();         // (what was there is read)
        stage_words<T>(words_of(a, layer) + a->at.inner, F / WORD, k0 / WORD, min(a->chunk, F - k0) / WORD, a->rows, down_rows(), pitch,
                       a->wait_most, lost);
        __syncthreads();
      },
      [&](float v0, float v1, int n, int m, const Two& t) {
        const f32x2 v = with_residual(a, v0, v1, t, stat2, m);
        const int at = m * W + n;
        if (layer + 1 < a->layers) publish_two(words_of(a, layer) + a->at.last + at, v.x, v.y);
        else *(f32x2*)(a->out + at) = v;
      });
  }
};

template <typename T, int ROWS, int SCD, int RQ, int RU>
__global__ void __launch_bounds__(THREADS, sizeof(T) == 2 ? 4 : 2) decode_layers_kernel(const Layers) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ float stat1[MOST_ROWS][2], stat2[MOST_ROWS][2];
  __shared__ Softmax sm;
  __shared__ Member joined;
  Args a = (Args)__builtin_amdgcn_kernarg_segment_ptr();
  if ((int)blockIdx.x >= a->blocks) {
    run_ahead<T>(a);
    return;
  }
  unsigned number = 0;
  if (threadIdx.x == 0) number = ask_in(a, 1);
  Block<T, ROWS, SCD, RQ, RU> block{smem, stat1, stat2, &sm, {}, {}, false, false};
  // (looked up meanwhile, as it is where all come)
  const int items = a->rows * (a->width / HD) * a->splits;
  block.mine = item_of<Kind<T>::KEYS>(a, min((int)blockIdx.x, items - 1));
#pragma unroll 1
  for (int m = 0; m < a->rows; ++m) block.cut |= shares_of(a->cached_lens[m], a->splits) > 1;
  if (threadIdx.x == 0) joined = join(a, number);
  __syncthreads();
  block.me = {__builtin_amdgcn_readfirstlane(joined.number), __builtin_amdgcn_readfirstlane(joined.of)};
  if (block.me.number < 0) return;
  if (block.me.number != (int)blockIdx.x) block.mine = item_of<Kind<T>::KEYS>(a, min(block.me.number, items - 1));
#pragma unroll 1
  for (int layer = 0; layer < a->layers; ++layer) {
    block.project(a, layer);
    block.put_out(a, layer);
    block.go_up(a, layer);
    block.go_down(a, layer);
  }
  if (block.lost) __hip_atomic_store(a->failed, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

// What a launch of these sizes is like: how often the keys of a request may be cut, how many of the inner width's elements lie in
// LDS at a time.
static int layer_blocks() { return max(1, tnx_compute_units() / 2); }
static int layer_splits(int rows, int width) { return max(1, min(8, layer_blocks() / (rows * (width / HD)))); }

constexpr int LDS_MOST = 72 * 1024;      // of a block, beside what the kernel has by name: two blocks a unit

static Places layer_places(int dtype, int rows, int width, int inner_width) {
  const int word = dtype == TNX_BF16 ? 2 : 1, splits = layer_splits(rows, width);
  Places p;
  p.qkv = 0;
  p.mixed = p.qkv + rows * (3 * width / word);
  p.inner = p.mixed + rows * (width / word);
  p.sum = p.inner + rows * (inner_width / word);
  p.last = p.sum + rows * width;
  p.parts = p.last + rows * width;
  p.all = p.parts + (splits > 1 ? rows * (width / HD) * splits * PART : 0);
  return p;
}

// The words of the layers' handoffs and, behind them, of `join`, all `NOT_YET` before the launch.
extern "C" int tnx_decode_layer_words(int dtype, int rows, int width, int inner_width, int layers) {
  if (rows <= 0 || rows > MOST_ROWS || width <= 0 || inner_width <= 0 || layers <= 0 || layers > MOST_LAYERS) return 0;
  return layers * layer_places(dtype, rows, width, inner_width).all + 2;
}

template <typename T, int ROWS, int SCD, int RQ, int RU>
static int launch_layers(Layers& a, hipStream_t stream) {
  const int size = (int)sizeof(T), turn = 128 * NW * SCD;
  const int room = LDS_MOST - red_bytes<T, 1>();
  int chunk = turn;
  while (chunk < a.inner_width && a.rows * (chunk + turn + Kind<T>::PAD) * size <= room) chunk += turn;
  a.chunk = min(chunk, a.inner_width);
  const int bytes = max(red_bytes<T, (RQ > RU ? RQ : RU)>() + a.rows * (a.width + Kind<T>::PAD) * size,
                        red_bytes<T, 1>() + a.rows * (a.chunk + Kind<T>::PAD) * size);
  TNX_REQUIRE(bytes <= LDS_MOST, "decode_layers: %d rows of %d want %d bytes of LDS", a.rows, a.width, bytes);
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void*)decode_layers_kernel<T, ROWS, SCD, RQ, RU>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_MOST);
    TNX_REQUIRE(e == hipSuccess, "decode_layers: cannot reserve %d bytes of LDS: %s", LDS_MOST, hipGetErrorString(e));
    configured = true;
  }
  a.blocks = layer_blocks();
  a.join_most = a.join_most ? min(a.join_most, a.blocks) : a.blocks;
  decode_layers_kernel<T, ROWS, SCD, RQ, RU><<<a.blocks + (a.blocks % 8 == 0 ? (sizeof(T) == 2 ? 32 : 96) : 0), THREADS, bytes, stream>>>(a);
  TNX_CHECK_LAUNCH("decode_layers");
  return 0;
}

// Consecutive layers; `words`: as many as `tnx_decode_layer_words` names. `join_most` 0: all blocks that come.
extern "C" int tnx_decode_layers(const Layers* layers, int dtype, hipStream_t stream) {
  Layers a = *layers;
  TNX_REQUIRE(a.rows > 0 && a.rows <= MOST_ROWS, "decode_layers: 1 to %d rows, got %d", MOST_ROWS, a.rows);
  TNX_REQUIRE(a.layers > 0 && a.layers <= MOST_LAYERS, "decode_layers: 1 to %d layers, got %d", MOST_LAYERS, a.layers);
  TNX_REQUIRE(a.width >= 128 && a.width <= 1024 && a.width % 128 == 0 && a.inner_width > 0 && a.inner_width % 128 == 0 && a.inner_width <= 4096,
              "decode_layers: widths in 128s up to 1,024, inner widths up to 4,096, got %d and %d", a.width, a.inner_width);
  TNX_REQUIRE(a.join_most >= 0 && a.wait_most > 0, "decode_layers: blocks that join and questions of a wait, got %d and %d", a.join_most, a.wait_most);
  TNX_REQUIRE(a.page_shift >= 6 && a.page_shift < 24 && a.table_width > 0 && a.num_pages > 0, "decode_layers: pages of a power of two from 64 keys on");
  TNX_REQUIRE(a.page_pad >= 0 && a.page_pad % 8 == 0, "decode_layers: bad distance between pages");
  TNX_REQUIRE(a.x && a.out && a.token_page && a.token_off && a.cached_lens && a.table && a.failed && a.words, "decode_layers: something is missing");
  TNX_REQUIRE(((uintptr_t)a.x | (uintptr_t)a.out | (uintptr_t)a.words) % 16 == 0, "decode_layers: the stream must be 16-byte aligned");
  for (int l = 0; l < a.layers; ++l) {
    const LayerOf& o = a.of[l];
    TNX_REQUIRE(o.w_qkv && o.w_out && o.w_up && o.w_down && o.b_qkv && o.b_out && o.b_up && o.b_down && o.first_weight && o.first_bias &&
                o.second_weight && o.second_bias && o.k_pages && o.v_pages, "decode_layers: something of layer %d is missing", l);
    TNX_REQUIRE(((uintptr_t)o.w_qkv | (uintptr_t)o.w_out | (uintptr_t)o.w_up | (uintptr_t)o.w_down | (uintptr_t)o.k_pages | (uintptr_t)o.v_pages |
                 (uintptr_t)o.b_qkv | (uintptr_t)o.b_out | (uintptr_t)o.b_up | (uintptr_t)o.b_down | (uintptr_t)o.first_weight | (uintptr_t)o.first_bias | (uintptr_t)o.second_weight | (uintptr_t)o.second_bias) % 16 == 0,
                "decode_layers: operands must be 16-byte aligned");
  }
  TNX_REQUIRE(a.out != a.x, "decode_layers: the result may not lie where the stream does");
  TNX_REQUIRE(dtype == TNX_F32 || dtype == TNX_BF16, "decode_layers: float32 or bfloat16");
  a.splits = layer_splits(a.rows, a.width);
  a.at = layer_places(dtype, a.rows, a.width, a.inner_width);
  if (dtype == TNX_BF16) return launch_layers<bf16_t, 8, 4, 3, 4>(a, stream);
  if (a.rows <= 4) return launch_layers<float, 4, 4, 3, 4>(a, stream);
  return launch_layers<float, 8, 2, 3, 2>(a, stream);
}
