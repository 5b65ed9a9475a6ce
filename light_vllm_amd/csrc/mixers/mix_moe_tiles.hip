// Mixture of experts on prompt steps, bf16: the experts' products as two grouped GEMMs on LDS tiles. The pairs are sorted
// by expert on the device as in mix_moe_gemm.hip, nothing is read back to the host, and no sorted copy of the activations
// is made: the first product gathers each token's row where it stages it.
//
// One workgroup sorted 65536 pairs in 68 us; the two launches here take 10.
//   moe_count_kernel   every workgroup counts the experts of its run of (token, choice) pairs and ranks its pairs
//   moe_place_kernel   every workgroup adds up the counts of the runs before its own and places its pairs; the first one
//                      lists the row tiles
//   moe_tile_kernel    C[row, n] = act(sum_k A[row, k] B_e[n, k]) on tiles of up to 256 x 256
#include "mix_common.h"

namespace lvmix {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((address_space(3))) uint8_t lds_u8;

constexpr int kTileRows = 256;
constexpr int kPlaceThreads = 1024;
constexpr int kRunPairs = 2048;      // pairs of a workgroup of the sort: two per thread
constexpr int kMostRuns = 64;        // beyond that the runs grow: every workgroup reads the counts of all of them

__global__ __launch_bounds__(kPlaceThreads) void moe_count_kernel(const int32_t* __restrict__ ids, int M, int E, int run,
                                                                   int32_t* __restrict__ inv, int32_t* __restrict__ counts) {
  extern __shared__ int32_t cnt[];   // [E]
  for (int e = threadIdx.x; e < E; e += kPlaceThreads) cnt[e] = 0;
  __syncthreads();
  const int64_t p0 = static_cast<int64_t>(blockIdx.x) * run;
  const int64_t p1 = p0 + run < M ? p0 + run : M;
  for (int64_t p = p0 + threadIdx.x; p < p1; p += kPlaceThreads) inv[p] = atomicAdd(&cnt[ids[p]], 1);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += kPlaceThreads) counts[static_cast<int64_t>(blockIdx.x) * E + e] = cnt[e];
}

__global__ __launch_bounds__(kPlaceThreads) void moe_place_kernel(const int32_t* __restrict__ ids, int M, int E, int run,
                                                                   const int32_t* __restrict__ counts,
                                                                   int32_t* __restrict__ sorted_pair, int32_t* __restrict__ inv,
                                                                   int32_t* __restrict__ tiles, int32_t* __restrict__ num_tiles,
                                                                   int max_tiles) {
  extern __shared__ int32_t sl[];
  int32_t* base = sl;                // [E] first row of this run's pairs
  int32_t* tot = sl + E;             // [E] pairs per expert
  int32_t* toff = sl + 2 * E;        // [E] first tile per expert
  const int runs = gridDim.x, mine = blockIdx.x;
  for (int e = threadIdx.x; e < E; e += kPlaceThreads) base[e] = tot[e] = 0;
  __syncthreads();
  // Bound by the wait for its loads. All threads share the counts: 32 experts in 32 runs take 5.5 us a launch, where a thread an
  // expert that went from run to run took 12.5.
  const int before = mine * E;
#pragma unroll 4
  for (int x = threadIdx.x; x < runs * E; x += kPlaceThreads) {
    const int n = counts[x], e = x % E;
    atomicAdd(&tot[e], n);
    if (x < before) atomicAdd(&base[e], n);
  }
  __syncthreads();
  if (threadIdx.x < kWave) {         // rows and tiles of the experts before each one: a scan of 64 experts at a time
    int rows = 0, tls = 0;
    for (int e0 = 0; e0 < E; e0 += kWave) {
      const int e = e0 + threadIdx.x;
      const int n = e < E ? tot[e] : 0, t = (n + kTileRows - 1) / kTileRows;
      int rn = n, rt = t;
      for (int o = 1; o < kWave; o <<= 1) {
        const int a = __shfl_up(rn, o, kWave), c = __shfl_up(rt, o, kWave);
        rn += static_cast<int>(threadIdx.x) >= o ? a : 0;
        rt += static_cast<int>(threadIdx.x) >= o ? c : 0;
      }
      if (e < E) {
        base[e] += rows + rn - n;
        toff[e] = tls + rt - t;
      }
      rows += __shfl(rn, kWave - 1, kWave);
      tls += __shfl(rt, kWave - 1, kWave);
    }
    if (mine == 0 && threadIdx.x == 0) num_tiles[0] = tls < max_tiles ? tls : max_tiles;
  }
  __syncthreads();
  const int64_t p0 = static_cast<int64_t>(mine) * run;
  const int64_t p1 = p0 + run < M ? p0 + run : M;
  for (int64_t p = p0 + threadIdx.x; p < p1; p += kPlaceThreads) {
    const int row = base[ids[p]] + inv[p];
    sorted_pair[row] = static_cast<int32_t>(p);
    inv[p] = row;
  }
  if (mine != 0) return;             // the first run's pairs open every expert: base is the expert's own first row there
  for (int e = threadIdx.x; e < E; e += kPlaceThreads) {
    const int n = tot[e];
    for (int j = 0, t = toff[e]; j * kTileRows < n && t < max_tiles; ++j, ++t) {
      tiles[3 * t] = e;
      tiles[3 * t + 1] = base[e] + j * kTileRows;
      tiles[3 * t + 2] = min(kTileRows, n - j * kTileRows);
    }
  }
}

struct MoeTileParams {
  const uint16_t* A;       // UP: activations [T, K]; else the sorted rows [M, K]
  const uint16_t* B;       // expert e's rows start at e * b_expert, row stride ldb
  uint16_t* C;             // [M, N] in sorted row order
  const int32_t *sorted_pair, *tiles, *num_tiles;
  int N, K, top, n_real;
  int64_t lda, ldb, ldc, b_expert;
  const float* row_scale;  // GLU: [pairs]
  float limit, alpha;
  int act;
  bool past;               // outputs do not stay in the caches: they are written past them
};

// Bound by the power that the products take: 16384 x 4096 x 4096 takes 404 us on 32 x 32 x 16 products and 376 on 16 x 16 x 32 ones, 290 both on zeros,
// and where a step's reads, barriers and requests stand moves neither. Half as many passes over the accumulators for the same products
// are what the smaller ones save (in a loop of products alone, without operands to bring, they are 5 % slower). The vendor's product takes 355 (265).
// 65536 rows through 2048 x 1536 and back, on 32 experts of 1940 to 2200 rows: the layer 888 -> 842 us. Other experts, launches in a graph, 32 x 32 x 16
// -> 16 x 16 x 32: 2048 x 1536, 32 experts, 4 each, 3000 tokens 212 -> 210, 7000 390 -> 362; 4096 x 3072, 6000 tokens 1225 -> 1150; gated units
// 2048 x 1536, 16384 tokens 1280 -> 1195; up to 64 rows an expert, where memory is the bound, level to 1 % (96 x 160, 16384 tokens 61 -> 52).
// Vendor GEMMs expert by expert took 1500 us for both, fragments straight from memory (moe_gemm_kernel) 3200.
//
// Four waves, one per SIMD: 64 MB rows x 256 columns of the product, each wave 32 MB x 128 of it in 64 MB accumulators. MB follows the
// tile's rows, so that an expert's last tile does no more products than its rows need (every expert has one: 5 % of the products above).
// A step over k is 64 wide, rows of 128 bytes, which is a cache line: with 64-byte rows every line was requested twice. The rows that the
// first product writes start at a line for the same reason (476 -> 436 us for the second). A step's operands lie in one of two LDS slots; the
// 16-byte piece c of row r sits at c ^ ((r >> 1) & 7), so that 16 neighbouring rows' pieces fill all banks once. The pieces come
// straight from memory (global_load_lds); the swizzle is applied to the address a lane loads from. A wave multiplies fragments that it read
// half a step before; 3/8 into a step everyone has read the rest of its slot, and the step after next is requested into it, spread over
// the remaining 5/8 and most of the second half: in a row behind one barrier, as many as the L1 takes 1024 clocks for, they held up the
// products behind them. The slots are arrays of their own so that the compiler knows which loads a read has to wait for.
// CHAIN (k in whole pairs of steps): a workgroup goes from tile to tile. The last two steps request the next tile's first two, which arrive while
// the outputs leave through LDS of their own, and nothing waits for a store until a step later; a tile by itself spent some 15 us on
// its way in and out. Other k drain the slots between tiles, and request the next tile's first steps in front of the outputs too (7000 tokens, 16 experts of
// 1024 x 352, 4 each: the layer's experts 112 -> 107 us, 107 with the tiles of 128 rows that came before; 16384 tokens 222 -> 217, 240).
// GLU: LDS rows 64 j .. 64 j + 31 of the weights hold gate columns 32 j .., the 32 after them the up columns of the same numbers.
template <bool UP, bool GLU, bool CHAIN, bool UNARY = false>
__global__ __launch_bounds__(256, 1) void moe_tile_kernel(MoeTileParams p) {
  static_assert((!GLU || UP) && (!UNARY || (UP && !GLU)), "gated units and activations follow the first product");
  constexpr int CW = GLU ? 128 : 256, WC = CW / 2;                   // output columns of a tile and of a wave
  constexpr int SLOT = 512 * 128, STAGE = 32 * WC * 2;               // bytes of a step's operands and of a wave's 32 output rows
  __shared__ __attribute__((aligned(1024))) uint8_t slot0[SLOT];
  __shared__ __attribute__((aligned(1024))) uint8_t slot1[SLOT];
  __shared__ __attribute__((aligned(1024))) uint8_t stage[4 * STAGE];

  // Workgroups go to the eight XCDs in turn; each XCD takes a run of neighbouring tiles (all columns of a few row tiles), whose operands its
  // L2 holds together, and its workgroups every so many-th of them. A last round that would leave half of them without work has its
  // tiles cut in two or four.
  const int ncol = (p.N + CW - 1) / CW;
  const int total = p.num_tiles[0] * ncol, per = (total + 7) / 8, begin = static_cast<int>(blockIdx.x & 7) * per;
  const int have = min(per, total - begin), stride = gridDim.x >> 3;
  if (have <= 0) return;
  const int whole = have / stride * stride, rest = have - whole, cut = 4 * rest <= stride ? 4 : (2 * rest <= stride ? 2 : 1);
  // by scalar loads: a vector load's wait would include the stores of the tile before
  const __attribute__((address_space(4))) int32_t* const tiles = (const __attribute__((address_space(4))) int32_t*)p.tiles;
  struct Tile { int q, e, row0, nrows, n0, col; };
  auto find = [&](int q) __attribute__((always_inline)) {            // the first of this workgroup's tiles from position q on; nrows 0: none is left
    Tile t{q, 0, 0, 0, 0, 0};
    for (; t.q < whole + rest * cut; t.q += stride) {
      const bool last = t.q >= whole;
      const int at = begin + (last ? whole + (t.q - whole) / cut : t.q), part = last ? (t.q - whole) % cut : 0;
      const int tile = at / ncol, size = kTileRows / cut;
      t.e = tiles[3 * tile];
      t.row0 = tiles[3 * tile + 1] + part * size;
      t.nrows = tiles[3 * tile + 2] - part * size;
      if (last) t.nrows = min(t.nrows, size);
      t.col = at % ncol;
      t.n0 = t.col * CW;
      if (t.e < p.n_real && t.nrows > 0) return t;
    }
    t.nrows = 0;
    return t;
  };
  Tile cur = find(blockIdx.x >> 3);
  if (cur.nrows == 0) return;

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = w & 1, wn = w >> 1;

  // the lane's number, unknown to the compiler: what is made of it for one tile is not kept in registers for all of them
  auto lane_here = [&]() __attribute__((always_inline)) {
    int x = lane;
    asm volatile("" : "+v"(x));
    return x;
  };
  // staging: one instruction brings 8 rows of 128 bytes
  const char *abase, *bbase;
  uint32_t aoff[8], boff[8];
  int pairs[8];                                                      // UP: (token, choice) of the rows that this lane stages
  int first;                                                         // where the walk over k begins
  auto look_up = [&](const Tile& t) __attribute__((always_inline)) {
    const int srow = lane_here() >> 3;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (UP) pairs[i] = p.sorted_pair[t.row0 + min(8 * (w + 4 * i) + srow, t.nrows - 1)];
  };
  const int full = p.K / 64;
  auto aim = [&](const Tile& t) __attribute__((always_inline)) {
    const int ln = lane_here(), srow = ln >> 3, spiece = (ln & 7) ^ (((w & 1) << 2) | ((ln >> 4) & 3));
    abase = reinterpret_cast<const char*>(UP ? p.A : p.A + static_cast<int64_t>(t.row0) * p.lda);
    bbase = reinterpret_cast<const char*>(p.B + static_cast<int64_t>(t.e) * p.b_expert + static_cast<int64_t>(t.n0) * p.ldb);
#pragma unroll
    for (int i = 0; i < 8; ++i) {                                    // rows past the tile's end repeat its last one; never stored
      const int src = UP ? pairs[i] / p.top : min(8 * (w + 4 * i) + srow, t.nrows - 1);
      aoff[i] = static_cast<uint32_t>(src) * static_cast<uint32_t>(2 * p.lda) + 16 * spiece;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int j = 8 * (w + 4 * i) + srow;
      const int n = min(t.n0 + (GLU ? (j >> 6) * 32 + (j & 31) : j), p.N - 1) - t.n0 + (GLU && (j & 32) ? p.N : 0);
      boff[i] = static_cast<uint32_t>(n) * static_cast<uint32_t>(2 * p.ldb) + 16 * spiece;
    }
    // Column tile j starts its walk over k further in and comes round: with every tile of an XCD at the same k the rows of a weight, whose
    // stride is a multiple of some KB, all come from one memory channel (second product of 65536 rows, 1536 x 2048: 511 us without, 436 with
    // 192 columns between neighbours; the first does not care). The order depends on the column alone, not on where the sort put a row.
    // Where k is an odd multiple of 32, its last half step ends the walk.
    first = full > 0 ? t.col * (UP ? 1 : 3) % full : 0;
  };
  // half a step: the pieces past the end repeat those in front of them
  const uint32_t back = ((lane & 7) ^ (((w & 1) << 2) | ((lane >> 4) & 3))) >= 4 ? 64u : 0u;
  auto place = [&](int c) __attribute__((always_inline)) {           // of step c in k: requests past the end repeat some step; never used
    const int at_k = c + first;
    return c < full ? (at_k < full ? at_k : at_k - full) : 64 * full < p.K ? full : 0;
  };
  auto load = [&](uint8_t* slot, int at_k, auto rows64, int x) __attribute__((always_inline)) {      // the x-th of a tile of 64 rows64
    const uint32_t less = !CHAIN && at_k == full ? back : 0u;
    lds_u8* const at = (lds_u8*)slot;
    constexpr int na = 2 * decltype(rows64)::value;
    const int i = x < na ? x : x - na;
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)((x < na ? abase : bbase) + 128 * static_cast<int64_t>(at_k) + ((x < na ? aoff[i] : boff[i]) - less)),
                                     (__attribute__((address_space(3))) void*)(at + (x < na ? 0 : 256 * 128) + 1024 * (w + 4 * i)), 16, 0, 0);
  };
  auto request = [&](uint8_t* slot, int c, auto rows64, int x) __attribute__((always_inline)) { load(slot, place(c), rows64, x); };
  using I4 = std::integral_constant<int, 4>;
  auto request_all = [&](uint8_t* slot, int c) __attribute__((always_inline)) {
    const int at_k = place(c);                                       // (once: asked for by every load it becomes three branches in front of each, 0.6 us a launch)
#pragma unroll
    for (int x = 0; x < 16; ++x) load(slot, at_k, I4{}, x);
  };
  // own LDS reads done, own requests landed (and stores on their way out); then everyone's
  auto turn = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(0x0070);
    asm volatile("s_barrier" ::: "memory");
  };

  look_up(cur);
  aim(cur);
  request_all(slot0, 0);
  request_all(slot1, 1);
  turn();
  // one tile of up to 64 MB rows, whose first two steps lie in the slots or (CHAIN) the second is on its way there
  auto tile = [&](auto mb) __attribute__((always_inline)) {
    constexpr int MB = decltype(mb)::value;
    constexpr int NB = 2 * MB, MUL = 8 * NB, READS = NB + 8, EARLY = MUL * 3 / 8;
    // fragments: lane l holds row l % 16 of a block, eight k from 8 (l / 16); half a step is 64 bytes across
    const int here = lane_here(), lr = here & 15, lq = here >> 4;
    const int fa0 = lr * 128 + ((lq ^ ((lr >> 1) & 7)) * 16) + wm * 32 * MB * 128;
    const int fb0 = lr * 128 + ((lq ^ ((lr >> 1) & 7)) * 16) + 256 * 128 + wn * 128 * 128;
    struct Frags { bf16x8_t a[NB], b[8]; };
    auto fetch = [&](const uint8_t* slot, int second, Frags& f, int x) __attribute__((always_inline)) {      // the x-th, in the products' order
      auto at = [&](int where) __attribute__((always_inline)) {
        return *reinterpret_cast<const __attribute__((address_space(3))) bf16x8_t*>((const lds_u8*)slot + where);
      };
      if (x == 0) f.b[0] = at(fb0 ^ (64 * second));
      else if (x <= NB) f.a[x - 1] = at((fa0 ^ (64 * second)) + 2048 * (x - 1));
      else f.b[x - NB] = at((fb0 ^ (64 * second)) + 2048 * (x - NB));
    };
    // The accumulators are tied to the accumulation registers: left to the compiler, 64 MB blocks of four are moved to and fro at every step.
    // It does not know of the products' latency then: what reads the sums stands behind eight other products or the wait in front of the output.
    f32x4_t acc[8][NB];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        asm volatile("" : "+a"(acc[i][j]));                          // (in front of the barrier, and so of the first product)
      }
    auto product = [&](const Frags& f, int i, int j) __attribute__((always_inline)) {
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(f.b[i]), "v"(f.a[j]));
    };
    Frags f0, f1;                                                    // first and second half of a step
    auto step = [&](uint8_t* mine, const uint8_t* next, int c, auto landed, auto more, auto rows64) __attribute__((always_inline)) {
      constexpr bool MORE = decltype(more)::value;
      constexpr int LOADS = 8 + 2 * decltype(rows64)::value, R1 = MORE ? LOADS * 3 / 8 : LOADS, R2 = LOADS - R1, LATE = MUL - EARLY;
#pragma unroll
      for (int q = 0; q < EARLY; ++q) {
        product(f0, q / NB, q % NB);
#pragma unroll
        for (int x = q * READS / EARLY; x < (q + 1) * READS / EARLY; ++x) fetch(mine, 1, f1, x);
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);                            // nobody reads this slot any more
      asm volatile("s_barrier" ::: "memory");
#pragma unroll
      for (int q = 0; q < LATE; ++q) {
        product(f0, (EARLY + q) / NB, q % NB);
#pragma unroll
        for (int x = q * R1 / LATE; x < (q + 1) * R1 / LATE; ++x) request(mine, c, rows64, x);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (MORE) {                                          // (otherwise f1's products are left to the output)
        if constexpr (!decltype(landed)::value) __builtin_amdgcn_s_waitcnt((R1 & 15) | ((R1 >> 4) << 14) | 0x0f70);
        asm volatile("s_barrier" ::: "memory");                      // the other one is complete
#pragma unroll
        for (int q = 0; q < MUL; ++q) {
          product(f1, q / NB, q % NB);
          if (q < EARLY) {
#pragma unroll
            for (int x = q * READS / EARLY; x < (q + 1) * READS / EARLY; ++x) fetch(next, 0, f0, x);
          }
#pragma unroll
          for (int x = q * R2 / MUL; x < (q + 1) * R2 / MUL; ++x) request(mine, c, rows64, R1 + x);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };

    Tile following;
    asm volatile("s_barrier" ::: "memory");                          // every wave's share of the first two steps has landed (awaited in front of its stores)
    // the rows' scales, asked for before a store is on its way: a load behind it would wait for it
    int who[GLU ? NB : 1];
    float rs[GLU ? NB : 1];
    if constexpr (GLU) {
#pragma unroll
      for (int j = 0; j < NB; ++j) who[j] = p.sorted_pair[cur.row0 + min(wm * 32 * MB + 16 * j + lr, cur.nrows - 1)];
    }
    auto scales = [&]() __attribute__((always_inline)) {
      if constexpr (GLU) {
#pragma unroll
        for (int j = 0; j < NB; ++j) rs[j] = p.row_scale[who[j]];
      }
    };
#pragma unroll
    for (int x = 0; x < READS; ++x) fetch(slot0, 0, f0, x);
    if constexpr (CHAIN) {
      following = find(cur.q + stride);
      if (following.nrows > 0) look_up(following);
      // (its first turn apart and without a condition: where it may be either, the compiler waits for loads that were requested behind it)
      step(slot0, slot1, 2, std::true_type{}, std::true_type{}, mb);
      step(slot1, slot0, 3, std::false_type{}, std::true_type{}, mb);
      scales();
      for (int c = 4; c < full; c += 2) {
        step(slot0, slot1, c, std::false_type{}, std::true_type{}, mb);
        step(slot1, slot0, c + 1, std::false_type{}, std::true_type{}, mb);
      }
      if (following.nrows > 0) aim(following);                       // the next tile's first two steps (or this one's, never used)
      step(slot0, slot1, 0, std::false_type{}, std::true_type{}, I4{});
      step(slot1, slot0, 1, std::false_type{}, std::false_type{}, I4{});
    } else {
      int c = 0;
      for (; c + 2 <= full; c += 2) {
        step(slot0, slot1, c + 2, std::false_type{}, std::true_type{}, mb);
        step(slot1, slot0, c + 3, std::false_type{}, std::true_type{}, mb);
      }
      if (c < full) step(slot0, slot1, c + 2, std::false_type{}, std::true_type{}, mb);
      if (64 * full < p.K) {
#pragma unroll
        for (int q = 0; q < MUL; ++q) product(f0, q / NB, q % NB);
      }
      following = find(cur.q + stride);
      scales();
      turn();                                                   // nobody reads or fills the slots any more
      if (following.nrows > 0) {
        look_up(following);
        aim(following);
        request_all(slot0, 0);
        request_all(slot1, 1);
      }
    }

    // Through the wave's own rows in LDS, 16 at a time in one of two places, so that they leave in whole lines. acc[i][j][u] is column
    // 16 i + 4 (lane / 16) + u of row 16 j + lane % 16. The eight bytes of a lane go to 16-byte piece c ^ swizzle(row).
    constexpr int PIECES = WC / 8, RPI = 64 / PIECES, PARTS = 16 / RPI, OUT = GLU ? 4 : 8;      // 16-byte pieces of a row; rows per store instruction
    auto swz = [&](int r) { return (PIECES == 16 ? r : r >> 1) & (PIECES - 1); };
    lds_u8* const mine = (lds_u8*)stage + w * STAGE;
    const int m0 = wm * 32 * MB, ln = lane_here(), er = ln & 15, eq = ln >> 4;
    typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
    auto put = [&](int j, int i) __attribute__((always_inline)) {    // columns 16 i .. of rows 16 j .. to their place
      const int src = GLU ? 4 * (i >> 1) + (i & 1) : i;
      asm volatile("" : "+a"(acc[src][j]));
      if constexpr (GLU) asm volatile("" : "+a"(acc[src + 2][j]));
      float v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if constexpr (GLU) {
          const float x = fminf(acc[src][j][u] * rs[j], p.limit);
          const float y = fminf(fmaxf(acc[src + 2][j][u] * rs[j], -p.limit), p.limit);
          v[u] = rs[j] != 0.0f ? x * sigmoidf_(p.alpha * x) * (y + 1.0f) : 0.0f;
        } else {
          v[u] = acc[src][j][u];
          if (UP && !UNARY) v[u] = v[u] < 0.0f ? 0.0f : v[u] * v[u];
        }
      }
      uint2 pair;
      pair.x = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{v[0], v[1]}), bf16x2_t));
      pair.y = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{v[2], v[3]}), bf16x2_t));
      const int piece = (2 * i + (eq >> 1)) ^ swz(er);
      *reinterpret_cast<__attribute__((address_space(3))) uint64_t*>(mine + (j & 1) * (STAGE / 2) + er * WC * 2 + piece * 16 + (((eq & 1) ^ (er >> 3)) & 1) * 8) =
          static_cast<uint64_t>(pair.x) | (static_cast<uint64_t>(pair.y) << 32);
    };
    auto leave = [&](int j, int i) __attribute__((always_inline)) {  // part i of rows 16 j ..
      const int r = i * RPI + ln / PIECES, c = ln % PIECES;
      const int n = cur.n0 + wn * WC + 8 * c;
      u32x4 v = *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(mine + (j & 1) * (STAGE / 2) + r * WC * 2 + (c ^ swz(r)) * 16);
      if (m0 + 16 * j + r >= cur.nrows || n >= p.N) return;          // N is a multiple of 8: a piece is in or out as a whole
      if ((r >> 3) & 1) v = u32x4{v[2], v[3], v[0], v[1]};
      if constexpr (UNARY) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          bf16_t lo, hi;
          stf(&lo, mix_act(__builtin_bit_cast(float, v[u] << 16), p.act));
          stf(&hi, mix_act(__builtin_bit_cast(float, v[u] & 0xffff0000u), p.act));
          v[u] = static_cast<uint32_t>(lo.bits) | (static_cast<uint32_t>(hi.bits) << 16);
        }
      }
      auto to = (__attribute__((address_space(1))) u32x4*)(p.C + static_cast<int64_t>(cur.row0 + m0 + 16 * j + r) * p.ldc + n);
      if (p.past) {
        asm volatile("" : "+v"(to));                                 // (keeps the two stores apart: as one they are both plain)
        __builtin_nontemporal_store(v, to);
        asm volatile("" ::: "memory");
      } else {
        *to = v;
      }
    };
    if constexpr (CHAIN) {                                           // the last half step
#pragma unroll
      for (int q = 0; q < MUL; ++q) product(f1, q / NB, q % NB);
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");               // the last sums are there
    __builtin_amdgcn_sched_barrier(0);
    // rows 16 (j + 1) go to LDS in front of the stores of rows 16 j
#pragma unroll
    for (int j = 0; j <= NB; ++j) {
      if (j < NB) {
#pragma unroll
        for (int i = 0; i < OUT; ++i) put(j, i);
      }
      if (j == 0) __builtin_amdgcn_s_waitcnt(0x0f70);                // the next tile's first two steps have landed: nothing there waits for a store
      if (j > 0 && !UNARY) {
#pragma unroll
        for (int i = 0; i < PARTS; ++i) leave(j - 1, i);
      } else if (j > 0) {
#pragma unroll 1
        for (int i = 0; i < PARTS; ++i) leave(j - 1, i);
      }
    }
    cur = following;
  };
  do {
    switch ((cur.nrows + 63) / 64) {
      case 1: tile(std::integral_constant<int, 1>{}); break;
      case 2: tile(std::integral_constant<int, 2>{}); break;
      case 3: tile(std::integral_constant<int, 3>{}); break;
      default: tile(std::integral_constant<int, 4>{}); break;
    }
  } while (cur.nrows > 0);
  __builtin_amdgcn_s_waitcnt(0x0070);                                // no request is on its way to this workgroup's LDS when it ends
}

}  // namespace lvmix

using namespace lvmix;

namespace {

int64_t most_tiles(int64_t pairs, int E) {
  const int64_t hit = pairs < E ? pairs : E;
  return pairs / kTileRows + hit;
}

int sort_runs(int64_t pairs) {
  const int64_t n = (pairs + kRunPairs - 1) / kRunPairs;
  return static_cast<int>(n < kMostRuns ? n : kMostRuns);
}

// sorted_pair [M] | inv [M] | counts [runs, E] | tiles [3 most] | num_tiles [1], in 32-bit words, padded to two cache lines so that the
// rows behind them start at one: steps of 128 bytes that lay across two lines cost the second product half as many requests again
int64_t index_words(int64_t M, int E) {
  return (2 * M + static_cast<int64_t>(sort_runs(M)) * E + 3 * most_tiles(M, E) + 1 + 63) / 64 * 64;
}

template <bool UP, bool GLU>
void tile_launch(const MoeTileParams& p, int64_t most, hipStream_t s) {
  const int64_t groups = 4 * most * ((p.N + (GLU ? 127 : 255)) / (GLU ? 128 : 256));      // one round: tiles may be cut in four
  const dim3 grid(static_cast<unsigned>(groups < 256 ? (groups + 7) / 8 * 8 : 256)), block(256);
  auto go = [&](auto unary) {
    constexpr bool U = decltype(unary)::value;
    if (p.K % 128 == 0 && p.K >= 256)
      moe_tile_kernel<UP, GLU, true, U><<<grid, block, 0, s>>>(p);
    else
      moe_tile_kernel<UP, GLU, false, U><<<grid, block, 0, s>>>(p);
  };
  if constexpr (UP && !GLU) {
    if (p.act != LV_MIX_ACT_RELU2) return go(std::true_type{});
  }
  go(std::false_type{});
}

}  // namespace

extern "C" {

int64_t lv_moe_tiled_workspace_bytes(int64_t T, int W, int F, int E, int top) {
  const int64_t M = T * top;
  return index_words(M, E) * 4 + ((M * F + 127) / 128 * 128 + M * W) * 2;
}

int lv_moe_tiled_ff(const void* h, const void* ids, const void* weights, const void* up_w, const void* down_w, int64_t down_ld,
                    void* out, void* workspace, int64_t T, int W, int F, int E_real, int n_through, int top, int act, int glu,
                    float limit, float alpha, void* stream) {
  if (T == 0) return 0;
  if (!h || !ids || !weights || !up_w || !down_w || !out || !workspace) return fail(-1, "lv_moe_tiled_ff: null pointer");
  const int64_t E = static_cast<int64_t>(E_real) + n_through;
  if (T < 0 || W <= 0 || F <= 0 || E_real <= 0 || n_through < 0 || top <= 0 || W % 32 != 0 || F % 32 != 0 || E > 4096 || act < 0 ||
      act > LV_MIX_ACT_GELU_TANH || (glu && n_through != 0))
    return fail(-1, "lv_moe_tiled_ff: width %d, expert size %d, %lld experts", W, F, (long long)E);
  if (down_ld <= 0) down_ld = static_cast<int64_t>(E_real) * F;
  if (down_ld < static_cast<int64_t>(E_real) * F || down_ld % 8 != 0 ||
      ((reinterpret_cast<uintptr_t>(h) | reinterpret_cast<uintptr_t>(up_w) | reinterpret_cast<uintptr_t>(down_w) |
        reinterpret_cast<uintptr_t>(workspace)) & 15) != 0)
    return fail(-1, "lv_moe_tiled_ff: row stride or alignment");
  const int64_t M = T * top;
  // offsets from a tile's first operand row are 32-bit byte counts
  const int64_t far = int64_t{1} << 31;
  if (M > (1 << 30) || T * W >= far || static_cast<int64_t>(F + 256) * W >= far || 256 * down_ld >= far ||
      256 * static_cast<int64_t>(F) >= far)
    return fail(-2, "lv_moe_tiled_ff: %lld rows of %d", (long long)T, W);
  const int64_t most = most_tiles(M, static_cast<int>(E));
  if (most * ((W + 127) / 128 + (F + 127) / 128) >= (1 << 30)) return fail(-2, "lv_moe_tiled_ff: %lld tiles", (long long)most);
  const int runs = sort_runs(M);
  const int run = static_cast<int>((M + runs - 1) / runs);
  int32_t* sorted_pair = static_cast<int32_t*>(workspace);
  int32_t* inv = sorted_pair + M;
  int32_t* counts = inv + M;
  int32_t* tiles = counts + static_cast<int64_t>(runs) * E;
  int32_t* num_tiles = tiles + 3 * most;
  uint16_t* mid = reinterpret_cast<uint16_t*>(sorted_pair + index_words(M, static_cast<int>(E)));
  uint16_t* rows = mid + (M * F + 127) / 128 * 128;
  hipStream_t s = as_stream(stream);
  const int32_t* pid = static_cast<const int32_t*>(ids);
  moe_count_kernel<<<dim3(runs), dim3(kPlaceThreads), sizeof(int32_t) * E, s>>>(pid, static_cast<int>(M), static_cast<int>(E), run, inv,
                                                                               counts);
  moe_place_kernel<<<dim3(runs), dim3(kPlaceThreads), 3 * sizeof(int32_t) * E, s>>>(
      pid, static_cast<int>(M), static_cast<int>(E), run, counts, sorted_pair, inv, tiles, num_tiles, static_cast<int>(most));
  // The operands of a tile's neighbours are what the L2s are for. Layers on 16384 tokens (201 and 268 MB) 855 us with outputs through them,
  // 845 past them; up to 6900 tokens (112 MB) the step behind finds some of them and reading them again takes 1 % longer.
  auto past = [&](int64_t width) { return M * width * 2 > int64_t{160} << 20; };
  MoeTileParams up{static_cast<const uint16_t*>(h), static_cast<const uint16_t*>(up_w), mid, sorted_pair, tiles, num_tiles,
                   F, W, top, E_real, W, W, F, static_cast<int64_t>(glu ? 2 : 1) * F * W,
                   static_cast<const float*>(weights), limit, alpha, act, past(F)};
  if (glu)
    tile_launch<true, true>(up, most, s);
  else
    tile_launch<true, false>(up, most, s);
  MoeTileParams down{mid, static_cast<const uint16_t*>(down_w), rows, sorted_pair, tiles, num_tiles,
                     W, F, top, E_real, F, down_ld, W, F, nullptr, 0.0f, 0.0f, 0, past(W)};
  tile_launch<false, false>(down, most, s);
  if (const int code = launched("lv_moe_tiled_ff")) return code;
  return lv_moe_combine_through(rows, inv, glu ? nullptr : weights, out, T, W, top, n_through > 0 ? ids : nullptr, E_real,
                                n_through > 0 ? h : nullptr, stream);
}

}  // extern "C"
