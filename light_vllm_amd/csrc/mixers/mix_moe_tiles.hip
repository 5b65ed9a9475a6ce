// Mixture of experts on prompt steps, bf16: the experts' products as two grouped GEMMs on LDS tiles. The pairs are sorted
// by expert on the device as in mix_moe_gemm.hip, nothing is read back to the host, and no sorted copy of the activations
// is made: the first product gathers each token's row where it stages it.
//
// One workgroup sorted 65536 pairs in 68 us; the two launches here take 19.
//   moe_count_kernel   every workgroup counts the experts of its run of (token, choice) pairs and ranks its pairs
//   moe_place_kernel   every workgroup adds up the counts of the runs before its own and places its pairs; the first one
//                      lists the row tiles
//   moe_tile_kernel    C[row, n] = act(sum_k A[row, k] B_e[n, k]) on a 256 x 256 or 128 x 256 tile
#include "mix_common.h"

namespace lvmix {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((address_space(3))) uint8_t lds_u8;

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

__global__ __launch_bounds__(kPlaceThreads) void moe_place_kernel(const int32_t* __restrict__ ids, int M, int E, int run, int BM,
                                                                   const int32_t* __restrict__ counts,
                                                                   int32_t* __restrict__ sorted_pair, int32_t* __restrict__ inv,
                                                                   int32_t* __restrict__ tiles, int32_t* __restrict__ num_tiles,
                                                                   int max_tiles) {
  extern __shared__ int32_t sl[];
  int32_t* base = sl;                // [E] first row of this run's pairs
  int32_t* tot = sl + E;             // [E] pairs per expert
  int32_t* toff = sl + 2 * E;        // [E] first tile per expert
  const int runs = gridDim.x, mine = blockIdx.x;
  for (int e = threadIdx.x; e < E; e += kPlaceThreads) {
    int before = 0, all = 0;
    for (int b = 0; b < runs; ++b) {
      const int n = counts[static_cast<int64_t>(b) * E + e];
      before += b < mine ? n : 0;
      all += n;
    }
    base[e] = before;
    tot[e] = all;
  }
  __syncthreads();
  if (threadIdx.x < kWave) {         // rows and tiles of the experts before each one: a scan of 64 experts at a time
    int rows = 0, tls = 0;
    for (int e0 = 0; e0 < E; e0 += kWave) {
      const int e = e0 + threadIdx.x;
      const int n = e < E ? tot[e] : 0, t = (n + BM - 1) / BM;
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
    for (int j = 0, t = toff[e]; j * BM < n && t < max_tiles; ++j, ++t) {
      tiles[3 * t] = e;
      tiles[3 * t + 1] = base[e] + j * BM;
      tiles[3 * t + 2] = min(BM, n - j * BM);
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
};

// Bound by the matrix cores at the rate that the card's power allows and by L2 on the way there: 65536 rows through 2048 x 1536
// and back 428 + 493 us = 964 and 836 TFLOP/s, where vendor GEMMs expert by expert took 1500 us for both (their grids of 48 to
// 64 tiles leave most of the chip idle) and fragments straight from memory (moe_gemm_kernel) 3200.
// Four waves, one per SIMD: 64 MB rows x 256 columns of the product, each wave 32 MB x 128 of it in 64 MB accumulators.
// A step over k is 32 wide. Its operands lie in one of four LDS slots, rows of 64 bytes; the 16-byte piece c of row r sits
// at c ^ ((r >> 2) & 3), so that 16 neighbouring rows' pieces fill all banks once. The pieces come straight from memory
// (global_load_lds); the swizzle is applied to the address a lane loads from. In step s a wave multiplies fragments that
// it read during step s - 1, reads those of step s + 1, and requests step s + 4 into the slot that step s was read from: one
// barrier a step, three steps for a load to arrive. The slots are arrays of their own so that the compiler knows which
// loads a read has to wait for.
// GLU: LDS rows 64 j .. 64 j + 31 hold gate columns 32 j .., the 32 after them the up columns of the same numbers.
template <int MB, bool UP, bool GLU>
__global__ __launch_bounds__(256, 1) void moe_tile_kernel(MoeTileParams p) {
  static_assert(!GLU || UP, "the gated unit follows the first product");
  constexpr int BM = 64 * MB, CW = GLU ? 128 : 256, WC = CW / 2;     // tile rows and output columns; a wave's output columns
  constexpr int SLOT = (BM + 256) * 64, LOADS = MB + 4;              // bytes of a slot; load instructions of a wave per step
  static_assert(32 * MB * WC * 2 <= SLOT, "a wave's output passes through one slot");
  __shared__ __attribute__((aligned(1024))) uint8_t slot0[SLOT];
  __shared__ __attribute__((aligned(1024))) uint8_t slot1[SLOT];
  __shared__ __attribute__((aligned(1024))) uint8_t slot2[SLOT];
  __shared__ __attribute__((aligned(1024))) uint8_t slot3[SLOT];

  // Workgroups go to the eight XCDs in turn; each XCD takes a run of neighbouring tiles (all columns of a few row tiles),
  // whose operands its L2 holds together.
  const int ncol = (p.N + CW - 1) / CW;
  const int total = p.num_tiles[0] * ncol, per = (total + 7) / 8;
  const int local = blockIdx.x >> 3;
  const int t = (blockIdx.x & 7) * per + local;
  if (local >= per || t >= total) return;
  const int tile = t / ncol, n0 = (t % ncol) * CW;
  const int e = p.tiles[3 * tile], row0 = p.tiles[3 * tile + 1], nrows = p.tiles[3 * tile + 2];
  if (e >= p.n_real) return;

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = w & 1, wn = w >> 1;

  // staging: one instruction brings 16 rows of 64 bytes
  const int srow = lane >> 2, spiece = (lane & 3) ^ ((lane >> 4) & 3);
  const char* const abase = reinterpret_cast<const char*>(UP ? p.A : p.A + static_cast<int64_t>(row0) * p.lda);
  const char* const bbase = reinterpret_cast<const char*>(p.B + static_cast<int64_t>(e) * p.b_expert + static_cast<int64_t>(n0) * p.ldb);
  uint32_t aoff[MB], boff[4];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int r = min(16 * (w + 4 * i) + srow, nrows - 1);           // rows past the tile's end repeat its last one; never stored
    const int src = UP ? p.sorted_pair[row0 + r] / p.top : r;
    aoff[i] = static_cast<uint32_t>(src) * static_cast<uint32_t>(2 * p.lda) + 16 * spiece;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = 16 * (w + 4 * i) + srow;
    const int n = min(n0 + (GLU ? (j >> 6) * 32 + (j & 31) : j), p.N - 1) - n0 + (GLU && (j & 32) ? p.N : 0);
    boff[i] = static_cast<uint32_t>(n) * static_cast<uint32_t>(2 * p.ldb) + 16 * spiece;
  }
  // Column tile j starts its walk over k further in and comes round: with every tile of an XCD at the same k the rows of a
  // weight, whose stride is a multiple of some KB, all come from one memory channel. The second product, whose weight rows
  // lie experts * ff apart, went from 745 to 493 us with 192 columns between neighbours (32 experts of 2048 x 1536, 65536
  // pairs), the first from 488 to 428 with 64. The order depends on the column alone, not on where the sort put a row.
  const int k0 = static_cast<int>(static_cast<int64_t>(t % ncol) * (UP ? 64 : 192) % p.K);
  auto request = [&](uint8_t* slot, int k) __attribute__((always_inline)) {
    int kk = (k < p.K ? k : 0) + k0;                                 // requests past the end repeat the first step; never used
    kk = kk < p.K ? kk : kk - p.K;
    lds_u8* const at = (lds_u8*)slot;
#pragma unroll
    for (int i = 0; i < MB; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(abase + 2 * static_cast<int64_t>(kk) + aoff[i]),
                                       (__attribute__((address_space(3))) void*)(at + 1024 * (w + 4 * i)), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(bbase + 2 * static_cast<int64_t>(kk) + boff[i]),
                                       (__attribute__((address_space(3))) void*)(at + BM * 64 + 1024 * (w + 4 * i)), 16, 0, 0);
  };

  // fragments: lane l holds row l % 32 of a block, eight k from 8 (l / 32); the second half of a step is 32 bytes across
  const int lr = lane & 31, lh = lane >> 5;
  const int fa0 = lr * 64 + ((lh ^ ((lr >> 2) & 3)) * 16) + wm * 32 * MB * 64;
  const int fb0 = lr * 64 + ((lh ^ ((lr >> 2) & 3)) * 16) + BM * 64 + wn * 128 * 64;
  const int fa1 = fa0 ^ 32, fb1 = fb0 ^ 32;
  struct Frags { bf16x8_t a[2][MB], b[2][4]; };
  auto fetch = [&](const uint8_t* slot, Frags& f) __attribute__((always_inline)) {
    const lds_u8* const at = (const lds_u8*)slot;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        f.b[h][i] = *reinterpret_cast<const __attribute__((address_space(3))) bf16x8_t*>(at + (h ? fb1 : fb0) + 2048 * i);
#pragma unroll
      for (int i = 0; i < MB; ++i)
        f.a[h][i] = *reinterpret_cast<const __attribute__((address_space(3))) bf16x8_t*>(at + (h ? fa1 : fa0) + 2048 * i);
    }
  };
  f32x16_t acc[4][MB];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // own requests of the next step landed (two later steps' may be on their way), own reads of this slot done; then everyone's
  auto turn = [&]() __attribute__((always_inline)) {
    constexpr int left = 2 * LOADS;
    __builtin_amdgcn_s_waitcnt((left & 15) | ((left >> 4) << 14) | 0x70);          // vmcnt(left) lgkmcnt(0)
    asm volatile("s_barrier" ::: "memory");
  };
  auto step = [&](uint8_t* freed, const uint8_t* next, int k, const Frags& cur, Frags& nxt) __attribute__((always_inline)) {
    turn();
    fetch(next, nxt);
    request(freed, k + 128);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur.b[h][i], cur.a[h][j], acc[i][j], 0, 0, 0);
    // reads behind the first products, then the requests; the products left at the end cover the last reads' way back
#pragma unroll
    for (int g = 0; g < 2 * LOADS; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (MB == 2 && g >= LOADS - 2 && g < 2 * LOADS - 2) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
    }
    if constexpr (MB == 4) {
#pragma unroll
      for (int g = 0; g < LOADS; ++g) {
        __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      }
    } else {
      __builtin_amdgcn_sched_group_barrier(0x008, 8 * MB - 2 * LOADS, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  request(slot0, 0);
  request(slot1, 32);
  request(slot2, 64);
  request(slot3, 96);
  Frags f0, f1;
  {
    constexpr int left = 3 * LOADS;
    __builtin_amdgcn_s_waitcnt((left & 15) | ((left >> 4) << 14) | 0x70);
    asm volatile("s_barrier" ::: "memory");
  }
  fetch(slot0, f0);
  int k = 0;                                                         // one way out of the loop: the wait counts stay exact
  for (; k + 128 <= p.K; k += 128) {
    step(slot0, slot1, k, f0, f1);
    step(slot1, slot2, k + 32, f1, f0);
    step(slot2, slot3, k + 64, f0, f1);
    step(slot3, slot0, k + 96, f1, f0);
  }
  if (k < p.K) {
    step(slot0, slot1, k, f0, f1);
    if (k + 32 < p.K) {
      step(slot1, slot2, k + 32, f1, f0);
      if (k + 64 < p.K) step(slot2, slot3, k + 64, f0, f1);
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0070);                                // the last requests have landed before the slots are used again
  asm volatile("s_barrier" ::: "memory");

  // Through the wave's own slot, so that rows leave in whole lines. acc[i][j][4 g + u] is column 32 i + 8 g + 4 lh + u of row
  // 32 j + lr. The eight bytes of a lane go to 16-byte piece c ^ swizzle(row), the two halves of a piece swapped in every
  // other block of 16 rows.
  constexpr int PIECES = WC / 8, RPI = 64 / PIECES;                  // 16-byte pieces of a row; rows per store instruction
  auto swz = [&](int r) { return (PIECES == 16 ? r : r >> 1) & (PIECES - 1); };
  lds_u8* const mine = (lds_u8*)(w == 0 ? slot0 : w == 1 ? slot1 : w == 2 ? slot2 : slot3);
  const int m0 = wm * 32 * MB;
#pragma unroll
  for (int j = 0; j < MB; ++j) {
    const int r = 32 * j + lr;
    float rs = 1.0f;
    if constexpr (GLU) rs = p.row_scale[p.sorted_pair[row0 + min(m0 + r, nrows - 1)]];
#pragma unroll
    for (int i = 0; i < (GLU ? 2 : 4); ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if constexpr (GLU) {
            const float x = fminf(acc[2 * i][j][4 * g + u] * rs, p.limit);
            const float y = fminf(fmaxf(acc[2 * i + 1][j][4 * g + u] * rs, -p.limit), p.limit);
            v[u] = rs != 0.0f ? x * sigmoidf_(p.alpha * x) * (y + 1.0f) : 0.0f;
          } else {
            v[u] = acc[i][j][4 * g + u];
            if (UP && p.act == LV_MIX_ACT_RELU2) v[u] = v[u] < 0.0f ? 0.0f : v[u] * v[u];
          }
        }
        uint32_t pair[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          bf16_t lo, hi;
          stf(&lo, v[2 * u]);
          stf(&hi, v[2 * u + 1]);
          pair[u] = static_cast<uint32_t>(lo.bits) | (static_cast<uint32_t>(hi.bits) << 16);
        }
        const int piece = (4 * i + g) ^ swz(r);
        *reinterpret_cast<__attribute__((address_space(3))) uint64_t*>(mine + r * WC * 2 + piece * 16 + ((lh ^ (r >> 4)) & 1) * 8) =
            static_cast<uint64_t>(pair[0]) | (static_cast<uint64_t>(pair[1]) << 32);
      }
  }
  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
#pragma unroll 2
  for (int i = 0; i < 32 * MB / RPI; ++i) {
    const int r = i * RPI + lane / PIECES, c = lane % PIECES;
    const int n = n0 + wn * WC + 8 * c;
    if (m0 + r >= nrows || n >= p.N) continue;                       // N is a multiple of 8: a piece is in or out as a whole
    u32x4 v = *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(mine + r * WC * 2 + (c ^ swz(r)) * 16);
    if ((r >> 4) & 1) v = u32x4{v[2], v[3], v[0], v[1]};
    if (UP && !GLU && p.act != LV_MIX_ACT_RELU2) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        bf16_t lo, hi;
        stf(&lo, mix_act(__builtin_bit_cast(float, v[u] << 16), p.act));
        stf(&hi, mix_act(__builtin_bit_cast(float, v[u] & 0xffff0000u), p.act));
        v[u] = static_cast<uint32_t>(lo.bits) | (static_cast<uint32_t>(hi.bits) << 16);
      }
    }
    *reinterpret_cast<u32x4*>(p.C + static_cast<int64_t>(row0 + m0 + r) * p.ldc + n) = v;
  }
}

}  // namespace lvmix

using namespace lvmix;

namespace {

// Rows of a tile. Below about a hundred rows an expert the taller tile is mostly padding and the shorter one's smaller
// staging wins (32 experts of 2048 x 1536: 109 against 118 us at 16 rows, 121 against 129 at 64); above, most experts need
// two short tiles and the taller one reads each weight half as often (145 against 178 us at 128 rows, 259 / 289 at 384,
// 1006 / 1168 at 2048; only right at 256, where half of the experts spill into a second tall tile, 246 against 214). Where all short
// tiles run at once, one a compute unit, the taller ones only leave more of the chip idle (8 experts of 1024 x 512 at 128 rows 54
// against 40 us, of 2048 x 1536 89 against 70); F in columns of 128, as gated units have them.
int tile_rows(int64_t pairs, int E, int W, int F) {
  const int64_t tiles = pairs / 128 + (pairs < E ? pairs : E);
  return pairs >= static_cast<int64_t>(E) * 96 && tiles * (((W > 2 * F ? W : 2 * F) + 255) / 256) > 256 ? 256 : 128;
}

int64_t most_tiles(int64_t pairs, int E, int BM) {
  const int64_t hit = pairs < E ? pairs : E;
  return pairs / BM + hit;
}

int sort_runs(int64_t pairs) {
  const int64_t n = (pairs + kRunPairs - 1) / kRunPairs;
  return static_cast<int>(n < kMostRuns ? n : kMostRuns);
}

// sorted_pair [M] | inv [M] | counts [runs, E] | tiles [3 most] | num_tiles [1], in 32-bit words, padded to 16 bytes
int64_t index_words(int64_t M, int E, int BM) {
  return (2 * M + static_cast<int64_t>(sort_runs(M)) * E + 3 * most_tiles(M, E, BM) + 1 + 3) / 4 * 4;
}

template <bool UP, bool GLU>
void tile_launch(const MoeTileParams& p, int64_t most, int BM, hipStream_t s) {
  const int64_t groups = most * ((p.N + (GLU ? 127 : 255)) / (GLU ? 128 : 256));
  const dim3 grid(static_cast<unsigned>((groups + 7) / 8 * 8));
  if (BM == 256)
    moe_tile_kernel<4, UP, GLU><<<grid, dim3(256), 0, s>>>(p);
  else
    moe_tile_kernel<2, UP, GLU><<<grid, dim3(256), 0, s>>>(p);
}

}  // namespace

extern "C" {

int64_t lv_moe_tiled_workspace_bytes(int64_t T, int W, int F, int E, int top) {
  const int64_t M = T * top;
  return index_words(M, E, tile_rows(M, E, W, F)) * 4 + M * (static_cast<int64_t>(F) + W) * 2;
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
  const int BM = tile_rows(M, static_cast<int>(E), W, F);
  const int64_t most = most_tiles(M, static_cast<int>(E), BM);
  if (most * ((W + 127) / 128 + (F + 127) / 128) >= (1 << 30)) return fail(-2, "lv_moe_tiled_ff: %lld tiles", (long long)most);
  const int runs = sort_runs(M);
  const int run = static_cast<int>((M + runs - 1) / runs);
  int32_t* sorted_pair = static_cast<int32_t*>(workspace);
  int32_t* inv = sorted_pair + M;
  int32_t* counts = inv + M;
  int32_t* tiles = counts + static_cast<int64_t>(runs) * E;
  int32_t* num_tiles = tiles + 3 * most;
  uint16_t* mid = reinterpret_cast<uint16_t*>(sorted_pair + index_words(M, static_cast<int>(E), BM));
  uint16_t* rows = mid + M * F;
  hipStream_t s = as_stream(stream);
  const int32_t* pid = static_cast<const int32_t*>(ids);
  moe_count_kernel<<<dim3(runs), dim3(kPlaceThreads), sizeof(int32_t) * E, s>>>(pid, static_cast<int>(M), static_cast<int>(E), run, inv,
                                                                               counts);
  moe_place_kernel<<<dim3(runs), dim3(kPlaceThreads), 3 * sizeof(int32_t) * E, s>>>(
      pid, static_cast<int>(M), static_cast<int>(E), run, BM, counts, sorted_pair, inv, tiles, num_tiles, static_cast<int>(most));
  MoeTileParams up{static_cast<const uint16_t*>(h), static_cast<const uint16_t*>(up_w), mid, sorted_pair, tiles, num_tiles,
                   F, W, top, E_real, W, W, F, static_cast<int64_t>(glu ? 2 : 1) * F * W,
                   static_cast<const float*>(weights), limit, alpha, act};
  if (glu)
    tile_launch<true, true>(up, most, BM, s);
  else
    tile_launch<true, false>(up, most, BM, s);
  MoeTileParams down{mid, static_cast<const uint16_t*>(down_w), rows, sorted_pair, tiles, num_tiles,
                     W, F, top, E_real, F, down_ld, W, F, nullptr, 0.0f, 0.0f, 0};
  tile_launch<false, false>(down, most, BM, s);
  if (const int code = launched("lv_moe_tiled_ff")) return code;
  return lv_moe_combine_through(rows, inv, glu ? nullptr : weights, out, T, W, top, n_through > 0 ? ids : nullptr, E_real,
                                n_through > 0 ? h : nullptr, stream);
}

}  // extern "C"
