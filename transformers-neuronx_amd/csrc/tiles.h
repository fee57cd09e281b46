// The inner loop of bfloat16 products by tiles (those of the experts): out[row][column] = sum over k of x[row][k] w[column][k] for a tile of TM rows by TN columns, by the
// waves of a block, with float32 sums.
#pragma once
#include "common.h"
#include <type_traits>

// A block of 2 x 2 waves, each of 32 MI rows by 32 NI columns as MI x NI MFMA 32x32x16 tiles: TM = 64 MI, TN = 64 NI.
// Both operands go from global memory straight into LDS in steps of 64 of K, ST stages deep; the 16-byte chunks of a row
// (8 of them, 128 bytes) lie swizzled by row, so that the fragment reads are free of bank conflicts.
// MI = NI = 2 and two stages take 64 KB and leave room for a second block on the compute unit, whose products cover this
// one's waits; where a unit has one block anyway, four stages (128 KB) do that instead.
template <int MI, int NI, int ST>
struct Tile {
  static constexpr int TM = 64 * MI, TN = 64 * NI;
  static constexpr int STAGE = (TM + TN) * 128;                     // bytes
  static constexpr int AHEAD = MI * NI <= 4 ? 4 : 2;
  static constexpr int LA = 2 * MI, LB = 2 * NI;                    // loads a wave issues for a step of x, of w
  static constexpr int OUT_ROW = 32 * NI * 4 + 16;                  // bytes of a row of the result on its way out
  static constexpr int OUT = 32 * OUT_ROW;                          // bytes of LDS a wave uses for that
  static constexpr int BYTES = ST * STAGE > 4 * OUT ? ST * STAGE : 4 * OUT;

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
  static __device__ __forceinline__ int row0() { return (wave() & 1) * 32 * MI; }
  static __device__ __forceinline__ int col0() { return (wave() >> 1) * 32 * NI; }

  // The sums over `steps` steps of 64 of K. A step's loads are issued one by one between the products of the step before:
  // a load takes the unit's address path for 16 cycles, and a wave waits where it comes to one that the others' loads
  // keep busy (all at the top of a step: 2 to 10 % slower).
  __device__ __forceinline__ void run(char* smem, const bf16_t* x, const bf16_t* w, int steps) {
    constexpr int L = LA + LB, P = 4 * MI * NI;                     // loads and products of a step
    const int lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
    const unsigned a_dst = lds_offset(smem) + LA * wave() * 1024, b_dst = lds_offset(smem) + TM * 128 + LB * wave() * 1024;
    auto load = [&](int t, int l) {
      const unsigned stage = (t % ST) * STAGE;
      if (l < LA) load_to_lds(x + (size_t)64 * t, xoff[l < LA ? l : 0], a_dst + stage + l * 1024);
      else load_to_lds(w + (size_t)64 * t, woff[l < LA ? 0 : l - LA], b_dst + stage + (l - LA) * 1024);
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
    auto step = [&](int t, auto with_loads) {
      constexpr bool more = decltype(with_loads)::value;
      // step t has landed when at most the loads of the ST - 2 steps behind it are still in flight
      const int ahead = min(ST - 2, steps - 1 - t);
      if (ST > 3 && ahead == 2) __builtin_amdgcn_s_waitcnt(0x0F70 | ((2 * L) & 15) | (((2 * L) >> 4) << 14));
      else if (ST > 2 && ahead == 1) __builtin_amdgcn_s_waitcnt(0x0F70 | (L & 15) | ((L >> 4) << 14));
      else __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
      const char* base = smem + (t % ST) * STAGE;
      bf16x8 a[4][MI], b[4][NI];
      auto frags = [&](int slot, int s) {
        const int chunk = ((2 * s + half) ^ swizzle) * 16;
#pragma unroll
        for (int i = 0; i < MI; ++i) a[slot][i] = *(const bf16x8*)(base + a0 + i * 4096 + chunk);
#pragma unroll
        for (int j = 0; j < NI; ++j) b[slot][j] = *(const bf16x8*)(base + b0 + j * 4096 + chunk);
      };
#pragma unroll
      for (int s = 0; s < AHEAD; ++s) frags(s, s);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s + AHEAD < 4) frags(s + AHEAD, s + AHEAD);      // later products' fragments arrive while these run
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[s][j], a[s][i], acc[i][j], 0, 0, 0);
            if constexpr (more) {
              const int q = (s * MI + i) * NI + j;
#pragma unroll
              for (int l = q * L / P; l < (q + 1) * L / P; ++l) {
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
  // several). `put(row, column, chunk)`: 16 bytes of the result, of type T, at a row and column of the wave's tile.
  template <typename T, int COLS, typename Value, typename Put>
  __device__ __forceinline__ void hand_out(char* smem, Value value, Put put) {
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
        put(32 * i + r, c * (16 / (int)sizeof(T)), *(const f32x4*)(mine + r * ROW + c * 16));
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
