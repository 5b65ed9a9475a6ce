// y [M, N] = x [M, K] w [N, K]^T for up to 64 rows of x, bf16 with f32 sums: the projections of a decode step.
//
// Bound by memory: the weights are read once, and every compute unit that takes part reads its share of them and the rows of x. What
// a compute unit takes in decides the time, so workgroups own few columns and all of k (nothing is summed across workgroups), and
// their eight waves share k between them: no value is fetched twice in a workgroup and no barrier stands in the loop. Weights and rows
// come as whole 128-byte lines, eight lanes a row, and pass through LDS of the wave's own into the matrix instructions' layout; loaded in
// that layout directly (sixteen rows of 64 bytes an instruction) the same launch took 14.9 us instead of 10.9 at 64 x 5152 x 2048. The
// row parts of one column tile are neighbours on one XCD, so the second reads the weights from its L2.
// A row's sums are formed in the same order whatever else is in the step and whatever tile it lands in.
//
// us in a replayed graph over weights that no cache holds, vendor product -> this, rows x columns x k: 1 x 5152 x 2048 12.3 -> 7.2,
// 16 x 2048 x 2048 11.0 -> 5.3, 32 x 8192 x 2048 13.2 -> 9.7, 64 x 5152 x 2048 12.9 -> 10.7, 64 x 2048 x 2048 11.7 -> 6.2,
// 64 x 4096 x 4096 15.2 -> 12.9, 8 x 10304 x 4096 26.3 -> 19.2, 16 x 5120 x 17408 115 -> 43. Not everywhere: 32 x 10304 x 4096 22.4 there,
// 25.3 here, 64 x 20480 x 4096 45 and 48. The caller's rule says where.
#include "mix_common.h"

namespace lvmix {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

constexpr int kRowsMax = 64;
constexpr int kRowsWaves = 8;
constexpr int kColumnsMax = 64;

struct RowsGemmParams {
  const uint16_t *x, *w;
  uint16_t* y;
  int64_t ldx, ldw, ldy;
  int M, N, K;
};

// A workgroup: 16 MT rows x 16 NT columns. PF pieces of 64 steps of k are on their way in registers. MANY: any number of rows, row tiles side by
// side on the grid, and all columns in each (those that a wide product leaves beside its tiles).
template <int MT, int NT, int PF, bool MANY = false>
__global__ __launch_bounds__(kRowsWaves * kWave) void rows_gemm_kernel(RowsGemmParams p) {
  constexpr int NW = kRowsWaves, RS = NT * 16 + 4;
  constexpr int STAGE = (MT + NT) * 2048, PART = MT * 16 * RS * 4, PER = STAGE > PART ? STAGE : PART;
  __shared__ __attribute__((aligned(16))) unsigned char lds[NW * PER];
  const int row_parts = (p.M + 16 * MT - 1) / (16 * MT);
  const int grp = blockIdx.x / (8 * row_parts), rem = blockIdx.x % (8 * row_parts);
  const int n0 = MANY ? 0 : (grp * 8 + rem % 8) * NT * 16, m0 = MANY ? blockIdx.x * MT * 16 : rem / 8 * MT * 16;
  if (n0 >= p.N) return;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, quad = lane >> 4;
  const int lrow = lane >> 3, lch = lane & 7;
  const int pieces = (p.K + 63) / 64, c0 = w * pieces / NW, c1 = (w + 1) * pieces / NW;
  unsigned char* mine = lds + w * PER;
  const uint16_t *wr[NT * 2], *xr[MT * 2];             // rows past the end repeat the last one; what they give is not stored
#pragma unroll
  for (int i = 0; i < NT * 2; ++i) wr[i] = p.w + min(n0 + 8 * i + lrow, p.N - 1) * p.ldw + 8 * lch;
#pragma unroll
  for (int i = 0; i < MT * 2; ++i) xr[i] = p.x + static_cast<int64_t>(min(m0 + 8 * i + lrow, p.M - 1)) * p.ldx + 8 * lch;
  u32x4_t wf[PF][NT * 2], xf[PF][MT * 2];
  f32x4_t acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  auto load = [&](int b, int c) __attribute__((always_inline)) {
    const int k = 64 * c + 32 < p.K || lch < 4 ? 64 * c : 64 * c - 32;         // k ends in the middle of a piece: its first half again
#pragma unroll
    for (int i = 0; i < NT * 2; ++i) wf[b][i] = *reinterpret_cast<const u32x4_t*>(wr[i] + k);
#pragma unroll
    for (int i = 0; i < MT * 2; ++i) xf[b][i] = *reinterpret_cast<const u32x4_t*>(xr[i] + k);
  };
  // 128 bytes a row; the 16-byte places of a row are permuted so that the reads of sixteen rows meet all banks
  auto put = [&](int i, u32x4_t v) __attribute__((always_inline)) {
    const int row = 8 * i + lrow;
    *reinterpret_cast<u32x4_t*>(mine + row * 128 + 16 * (lch ^ ((row >> 1) & 7))) = v;
  };
  auto get = [&](int t, int half) __attribute__((always_inline)) {
    const int row = 16 * t + r;
    return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(mine + row * 128 + 16 * ((4 * half + quad) ^ ((row >> 1) & 7))));
  };
#pragma unroll
  for (int b = 0; b < PF; ++b)
    if (c0 + b < c1) load(b, c0 + b);
  for (int c = c0; c < c1; c += PF) {
#pragma unroll
    for (int b = 0; b < PF; ++b) {
      if (c + b >= c1) break;
#pragma unroll
      for (int i = 0; i < MT * 2; ++i) put(i, xf[b][i]);
#pragma unroll
      for (int i = 0; i < NT * 2; ++i) put(MT * 2 + i, wf[b][i]);
      __builtin_amdgcn_wave_barrier();                 // the wave's own LDS: its operations are carried out in order
      bf16x8_t xv[MT][2], wv[NT][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < MT; ++i) xv[i][h] = get(i, h);
#pragma unroll
        for (int i = 0; i < NT; ++i) wv[i][h] = get(MT + i, h);
      }
      __builtin_amdgcn_wave_barrier();
      if (c + b + PF < c1) load(b, c + b + PF);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (h == 1 && 64 * (c + b) + 32 >= p.K) break;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
          for (int j = 0; j < MT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[i][h], xv[j][h], acc[i][j], 0, 0, 0);
      }
    }
  }
  // the waves' sums, one behind the other
  __builtin_amdgcn_wave_barrier();
  float* part = reinterpret_cast<float*>(mine);
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) *reinterpret_cast<f32x4_t*>(part + (16 * j + r) * RS + 16 * i + 4 * quad) = acc[i][j];
  __syncthreads();
  for (int e = threadIdx.x; e < MT * 16 * NT * 4; e += NW * kWave) {
    const int m = e / (NT * 4), n = e % (NT * 4) * 4;
    float4 s{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const float4 t = ld4(reinterpret_cast<const float*>(lds + i * PER) + m * RS + n);
      s = float4{s.x + t.x, s.y + t.y, s.z + t.z, s.w + t.w};
    }
    if (m0 + m >= p.M) continue;
    bf16_t* to = reinterpret_cast<bf16_t*>(p.y) + static_cast<int64_t>(m0 + m) * p.ldy + n0 + n;
    if (n0 + n + 3 < p.N && p.ldy % 4 == 0) {
      st4(to, s);
    } else {
      const float v[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n0 + n + i < p.N) stf(to + i, v[i]);
    }
  }
}

static int rows_gemm_groups(const RowsGemmParams& p, int mt, int nt) {
  return ((p.N + 16 * nt - 1) / (16 * nt) + 7) / 8 * 8 * ((p.M + 16 * mt - 1) / (16 * mt));
}

template <int MT, int NT>
static void rows_gemm_launch(const RowsGemmParams& p, hipStream_t s) {
  rows_gemm_kernel<MT, NT, NT == 1 ? 2 : 1><<<dim3(rows_gemm_groups(p, MT, NT)), dim3(kRowsWaves * kWave), 0, s>>>(p);
}

}  // namespace lvmix

using namespace lvmix;

extern "C" int lv_rows_gemm(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y, int64_t ldy, int M, int N, int K,
                            void* stream) {
  if (M == 0 || N == 0) return 0;
  if (!x || !w || !y) return fail(-1, "lv_rows_gemm: null pointer");
  if (M < 0 || M > kRowsMax || N < 0 || K <= 0 || K % 32 != 0) return fail(-1, "lv_rows_gemm: bad sizes");
  if (ldx < 0 || ldx % 8 != 0 || ldw < K || ldw % 8 != 0 || ldy < N || reinterpret_cast<uintptr_t>(x) % 16 != 0 ||
      reinterpret_cast<uintptr_t>(w) % 16 != 0 || reinterpret_cast<uintptr_t>(y) % 8 != 0)
    return fail(-1, "lv_rows_gemm: strides or alignment");
  RowsGemmParams p{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), static_cast<uint16_t*>(y), ldx, ldw, ldy, M, N, K};
  // The tile that brings the least into a compute unit: rounds of 256 workgroups times a workgroup's rows of x and w. us at
  // 64 x 2592 x 2048 (rows x columns of a tile): 32 x 32 7.6, 16 x 16 8.9; at 64 x 5152 x 2048 64 x 32 10.9, 16 x 32 12.2, 32 x 32 12.3; at
  // 48 x 2048 x 2048 16 x 32 6.3, 16 x 16 6.7. Tiles of more rows by 16 columns never count less than one of these (32 x 16 as much as 16 x 32,
  // though it took 5.8 at the last), so there are none.
  auto count = [&](int mt, int nt) { return (rows_gemm_groups(p, mt, nt) + 255) / 256 * (mt + nt); };
  int best = 0, least = count(1, 1);
  for (int mt = 1; mt <= (M + 15) / 16; ++mt)
    if (count(mt, 2) < least) {
      best = mt;
      least = count(mt, 2);
    }
  hipStream_t s = as_stream(stream);
  switch (best) {
    case 0: rows_gemm_launch<1, 1>(p, s); break;
    case 1: rows_gemm_launch<1, 2>(p, s); break;
    case 2: rows_gemm_launch<2, 2>(p, s); break;
    case 3: rows_gemm_launch<3, 2>(p, s); break;
    default: rows_gemm_launch<4, 2>(p, s);
  }
  return launched("lv_rows_gemm");
}

// Few columns of many rows, bound by reading x once (16384 x 2048 in 12.8 us, 5.2 TB/s, for 32 columns, 13.4 for 16, 16.3 for 64, of which the
// rows of w that every workgroup reads are the rest): 32 rows a workgroup, eight waves share k, and all the columns in one, so that x is not
// read twice. The vendor's product of 5152 columns instead of 5120 takes 42 us more (232 -> 274).
extern "C" int lv_columns_gemm(const void* x, int64_t ldx, const void* w, int64_t ldw, void* y, int64_t ldy, int64_t M, int N, int K,
                               void* stream) {
  if (M == 0 || N == 0) return 0;
  if (!x || !w || !y) return fail(-1, "lv_columns_gemm: null pointer");
  if (M < 0 || M > (int64_t{1} << 30) || N < 0 || N > kColumnsMax || K <= 0 || K % 32 != 0) return fail(-1, "lv_columns_gemm: bad sizes");
  if (ldx < K || ldx % 8 != 0 || ldw < K || ldw % 8 != 0 || ldy < N || reinterpret_cast<uintptr_t>(x) % 16 != 0 ||
      reinterpret_cast<uintptr_t>(w) % 16 != 0 || reinterpret_cast<uintptr_t>(y) % 8 != 0)
    return fail(-1, "lv_columns_gemm: strides or alignment");
  const RowsGemmParams p{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), static_cast<uint16_t*>(y), ldx, ldw, ldy,
                         static_cast<int>(M), N, K};
  hipStream_t s = as_stream(stream);
  const dim3 block(kRowsWaves * kWave);
  const unsigned rows = static_cast<unsigned>((M + 31) / 32);
  if (N <= 16) rows_gemm_kernel<2, 1, 2, true><<<dim3(rows), block, 0, s>>>(p);
  else if (N <= 32) rows_gemm_kernel<2, 2, 1, true><<<dim3(rows), block, 0, s>>>(p);
  else rows_gemm_kernel<2, 4, 1, true><<<dim3(rows), block, 0, s>>>(p);
  return launched("lv_columns_gemm");
}
