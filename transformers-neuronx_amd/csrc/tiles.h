// The inner loop of bfloat16 products by tiles (plain ones in `gemm.hip`, those of the experts): out[row][column] = sum over k
// of x[row][k] w[column][k] for a tile of TM rows by TN columns, by the waves of a block, with float32 sums.
#pragma once
#include "common.h"
#include <type_traits>

// A block of WM x WN waves, each of 32 MI rows by 32 NI columns as MI x NI MFMA 32x32x16 tiles: TM = 32 MI WM, TN = 32 NI WN.
// Both operands go from global memory straight into LDS in steps of 64 of K, ST stages deep; the 16-byte chunks of a row
// (8 of them, 128 bytes) lie swizzled by row, so that the fragment reads are free of bank conflicts.
// Eight waves give every matrix core two: one multiplies while the other waits for LDS or for a load to be taken. Measured as a
// plain product of 2,048 rows, 4,096 columns, K 16,384, us (TFLOP/s): four waves of 128 x 64 on 256 x 128, three stages, 264
// (1,040); eight of 64 x 64 there 243 (1,130), with the next step's fragments read before the last products of a step 235
// (1,170); four of 64 x 64 on 128 x 128, two stages and two blocks a unit, 306; 256 x 256, two stages, 263 at best.
template <int MI, int NI, int ST, int WM = 2, int WN = 2>
struct Tile {
  static constexpr int WAVES = WM * WN, TM = 32 * MI * WM, TN = 32 * NI * WN;
  static constexpr int STAGE = (TM + TN) * 128;                     // bytes
  static constexpr int LA = TM / 8 / WAVES, LB = TN / 8 / WAVES;    // loads a wave issues for a step of x, of w
  static constexpr int OUT_ROW = 32 * NI * 4 + 16;                  // bytes of a row of the result on its way out
  static constexpr int OUT = 32 * OUT_ROW;                          // bytes of LDS a wave uses for that
  static constexpr int BYTES = ST * STAGE > WAVES * OUT ? ST * STAGE : WAVES * OUT;

  // what this lane loads at step 0, as bytes from the operands' beginnings (operands of less than 4 GB): set by the
  // caller from `x_row` / `w_row` and `k_of`
  unsigned xoff[LA], woff[LB];
  f32x16 acc[MI][NI];         // element e of a lane: row lane % 32, column 8 (e / 4) + 4 (lane / 32) + e % 4 of the 32 x 32

  static __device__ __forceinline__ int wave() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }
  // the row of the tile of x (column of w) that load j of this lane belongs to, and the first of its 8 elements of K
  static __device__ __forceinline__ int x_row(int j) { return (LA * wave() + j) * 8 + ((threadIdx.x & 63) >> 3); }
  static __device__ __forceinline__ int w_row(int j) { return (LB * wave() + j) * 8 + ((threadIdx.x & 63) >> 3); }
  static __device__ __forceinline__ int k_of(int row) { return 8 * ((threadIdx.x & 7) ^ ((row >> 1) & 7)); }
  // the first row and column of this wave within the tile
  static __device__ __forceinline__ int row0() { return (wave() % WM) * 32 * MI; }
  static __device__ __forceinline__ int col0() { return (wave() / WM) * 32 * NI; }

  // The sums over `steps` steps of 64 of K. A step is four products of 16 of K; its loads, for the step ST - 1 ahead, are
  // issued one by one between them. The wait for the next step's operands and the block's meeting come before the last of
  // the four, and so do the reads of the next step's first fragments: those products run while the fragments arrive, where
  // after a meeting at the top of a step the matrix unit would stand until LDS has answered.
  __device__ __forceinline__ void run(char* smem, const bf16_t* x, const bf16_t* w, int steps) {
    constexpr int L = LA + LB, P = 3 * MI * NI;                     // loads of a step, and the products they stand between
    const int lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
    const unsigned a_dst = lds_offset(smem) + LA * wave() * 1024, b_dst = lds_offset(smem) + TM * 128 + LB * wave() * 1024;
    auto load = [&](int t, int l) {
      const unsigned stage = (t % ST) * STAGE;
      if (l < LA) load_to_lds(x + (size_t)64 * t, xoff[l < LA ? l : 0], a_dst + stage + l * 1024);
      else load_to_lds(w + (size_t)64 * t, woff[l < LA ? 0 : l - LA], b_dst + stage + (l - LA) * 1024);
    };
    // step t has landed when at most the loads of the `behind` steps after it are still in flight
    auto landed = [&](int behind) {
      if (ST > 4 && behind >= 3) __builtin_amdgcn_s_waitcnt(0x0F70 | ((3 * L) & 15) | (((3 * L) >> 4) << 14));
      else if (ST > 3 && behind == 2) __builtin_amdgcn_s_waitcnt(0x0F70 | ((2 * L) & 15) | (((2 * L) >> 4) << 14));
      else if (ST > 2 && behind == 1) __builtin_amdgcn_s_waitcnt(0x0F70 | (L & 15) | ((L >> 4) << 14));
      else __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
    };
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
#pragma unroll
    for (int p = 0; p < ST - 1; ++p)
      if (p < steps) {
#pragma unroll
        for (int l = 0; l < L; ++l) load(p, l);
      }
    const int swizzle = (l32 >> 1) & 7;
    const int a0 = (row0() + l32) * 128, b0 = TM * 128 + (col0() + l32) * 128;
    bf16x8 a[4][MI], b[4][NI];
    auto frags = [&](int t, int s) {
      const char* base = smem + (t % ST) * STAGE;
      const int chunk = ((2 * s + half) ^ swizzle) * 16;
#pragma unroll
      for (int i = 0; i < MI; ++i) a[s][i] = *(const bf16x8*)(base + a0 + i * 4096 + chunk);
#pragma unroll
      for (int j = 0; j < NI; ++j) b[s][j] = *(const bf16x8*)(base + b0 + j * 4096 + chunk);
    };
    landed(min(ST - 2, steps - 1));
    frags(0, 0);
    auto step = [&](int t, auto with_loads) {
      constexpr bool more = decltype(with_loads)::value;
#pragma unroll
      for (int s = 1; s < 4; ++s) frags(t, s);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s == 3 && (more || t + 1 < steps)) {
          landed(more ? ST - 2 : min(ST - 2, steps - 2 - t));
          frags(t + 1, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[s][j], a[s][i], acc[i][j], 0, 0, 0);
            if constexpr (more) {
              const int q = (s * MI + i) * NI + j;
#pragma unroll
              for (int l = q * L / P; l < (q + 1) * L / P && l < L; ++l) {
                __builtin_amdgcn_sched_barrier(0);
                load(t + ST - 1, l);
                __builtin_amdgcn_sched_barrier(0);
              }
            }
          }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    int t = 0;
    for (; t + ST - 1 < steps; ++t) step(t, std::true_type{});
    for (; t < steps; ++t) step(t, std::false_type{});
    __syncthreads();      // the stages are free: the result may go through them
  }

  // Hands the result over by rows. `value(i, j, e, row, column)`: the element as it goes out (row and column of the tile,
  // j and e of the accumulator); COLS columns of a wave go out (all 32 NI, or the first 32 j = 0 where `value` joins
  // several). `put(row, column, chunk, k)`: 16 bytes of the result, of type T, at a row and column of the wave's tile, the lane's
  // k-th (`out_row`, `out_column`: where that is).
  template <typename T, int COLS>
  static constexpr int out_count() { return MI * 32 * COLS * (int)sizeof(T) / 16 / 64; }
  template <typename T, int COLS>
  static __device__ __forceinline__ int out_row(int k) {
    constexpr int CHUNKS = COLS * (int)sizeof(T) / 16;
    return k * (64 / CHUNKS) + (int)(threadIdx.x & 63) / CHUNKS;
  }
  template <typename T, int COLS>
  static __device__ __forceinline__ int out_column() {
    constexpr int CHUNKS = COLS * (int)sizeof(T) / 16;
    return (int)(threadIdx.x & 63) % CHUNKS * (16 / (int)sizeof(T));
  }
  template <typename T, int COLS, typename Value, typename Put>
  static __device__ __forceinline__ void hand_out(char* smem, Value value, Put put) {
    const int lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
    constexpr int ROW = COLS * (int)sizeof(T) + 16;
    char* mine = smem + wave() * OUT;
    typedef T four __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
      for (int j = 0; j < COLS / 32; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int c = 32 * j + 8 * g + 4 * half;
          four v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = (T)value(i, j, 4 * g + e, 32 * i + l32, c + e);
          *(four*)(mine + l32 * ROW + c * (int)sizeof(T)) = v;
        }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      constexpr int CHUNKS = COLS * (int)sizeof(T) / 16, PASS = 64 / CHUNKS;
#pragma unroll
      for (int r0 = 0; r0 < 32; r0 += PASS) {
        const int r = r0 + lane / CHUNKS, c = lane % CHUNKS;
        put(32 * i + r, c * (16 / (int)sizeof(T)), *(const f32x4*)(mine + r * ROW + c * 16), (32 * i + r0) / PASS);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
};

// The place of a block among `count`, so that the blocks of one XCD (every eighth block) are neighbours.
__device__ __forceinline__ int by_xcd(int block, int count) {
  const int xcd = block & 7, each = count >> 3, more = count & 7;
  return xcd * each + min(xcd, more) + (block >> 3);
}
