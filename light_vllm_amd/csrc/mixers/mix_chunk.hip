// Recurrences with one decay per head and token, 32 tokens at a time on the f32 matrix instructions.
//
//   S_t = g_t S_(t-1) + k_t u_t^T,   o_t = S_t^T q_t,   u_t = w_t v_t                          (step sizes, constant decays)
//                                                       u_t = beta_t (v_t - g_t S_(t-1)^T k_t)  (delta rule)
//
// With G_t the product of a chunk's decays up to t, E_t the product of those behind t, D_tj = g_(j+1) .. g_t and S the state
// in front of the chunk:
//
//   U = V                       (delta rule: U = T (V - diag(G) K S),  T = (I + tril(diag(beta) (D o K K^T), -1))^-1 diag(beta))
//   O = diag(G) Q S + P U,      P_tj = D_tj (q_t . k_j) w_j for j <= t   (w = 1 for the delta rule)
//   S <- G_last S + K^T diag(E w) U
//
// chunk_prep_kernel      T, P, G and E w of every chunk, all of them side by side (constant decays may form them in the scan: chunk_own)
// chunk_scan_kernel      the chain over a sequence's chunks; a wave owns all D rows of 16 columns of the state
// chunk_step_kernel      the same for step sizes, on the bf16 matrix instructions
// chunk_combine_kernel   starting states of a sequence's segments, where there are too few sequences for the chip
//
// Every product of decays is formed as one (no exponentials of differences of logarithms), so a ratio is as exact as in the
// token loop and a decay of zero stays zero.
//
// Products are f32 with f32 sums, as in the token loop: v_mfma_f32_16x16x4_f32 in the scan, v_mfma_f32_32x32x2_f32 in front of it (the
// delta rule's q k^T in 64 bits). The 16 x 16 result layout (4 registers, rows 4 (lane / 16) + i, column lane % 16) is its own
// right-hand operand layout if step i multiplies the left-hand column of the same number: the state, U and V - G K S go from product
// to product in registers, and only q, k, T and P pass through LDS.
//
// Bound by the chain of a chunk, two waves a SIMD: 2 D Dv + 24 Dv multiply-adds a token and head at the f32 matrix rate (3 D Dv + 48 Dv
// for the delta rule), and beside them the vector ALU's work of staging the next chunk, which stands among the last products without a
// branch between. The token loop they replace did fewer operations, but on the vector ALU, one token behind the other. Kernels of a
// layer, us, token loop -> f32 chunks -> staged among the products / on bf16 instructions: 16 x 1024 tokens, delta rule (16 heads, 128 x
// 128) 993 -> 377 -> 343; constant decays (16 heads, 128 x 128) 596 -> 295 -> 281; step sizes (32 heads, 128 x 64; 7 prompts, the longest
// 3750) 1531 -> 456 -> 323, 314 with three waves a SIMD in front of the scan. Pieces for all products of the other two kinds, whose q, k and v are f32, were built and gained nothing: six to eight
// products for one, and every row to cut.
#include "mix_common.h"

#include <algorithm>

namespace lvmix {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef __bf16 chunk_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 chunk_bf16x4 __attribute__((ext_vector_type(4)));
constexpr int kCh = 32;               // tokens of a chunk
constexpr int kPad = 4;               // floats behind every LDS row: 16-byte reads of 8 rows meet 8 different bank groups

enum ChunkKind { kChunkStep = LV_MIX_CHUNK_STEP, kChunkConst = LV_MIX_CHUNK_CONST, kChunkDelta = LV_MIX_CHUNK_DELTA };

struct ChunkParams {
  const void *q, *k, *v;              // act rows of stride ldq, ldk, ldv: query/key group h / (H/G) of D, value head h of Dv
  int64_t ldq, ldk, ldv;
  const void* a;                      // step sizes: act rows of stride lda; delta rule: beta f32 [T, H]
  int64_t lda;
  const float* decay;                 // [H] (constant) or [T, H] (delta rule)
  const float *p0, *p1, *p2;          // step sizes: bias, log rate, skip [H]
  float* state;
  const int32_t *cu_q, *ctx_lens, *slots;
  float* o;
  float *P, *Tm, *Gf, *Ef;            // workspace: [T, H, 32], [T, H, 32] (delta rule), [T, H], [T, H]
  float *seg_state, *seg_decay;       // workspace: [B, segments, H, D, Dv], [B, segments, H]
  int B, H, G, D, Dv, seg_len, segs;
  // norm and gate behind the read-out: o is then the layer's act rows [T, H * Dv]
  const bf16_t* gate;                 // rows of stride ld_gate
  int64_t ld_gate;
  const float* norm_w;                // [Dv]
  float eps;
  int gate_silu;                      // silu, else sigmoid
};

__device__ __forceinline__ float chunk_lane(float x, int i) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), i));
}
__device__ __forceinline__ int acc_row(int i, int half) { return 8 * (i >> 2) + 4 * half + (i & 3); }

template <bool SILU>
__device__ __forceinline__ float4 chunk_act(float4 x) {
  if constexpr (SILU) return float4{quick_silu_(x.x), quick_silu_(x.y), quick_silu_(x.z), quick_silu_(x.w)};
  return x;
}

// grid: (chunks, groups), four waves. The chunks of all sequences lie side by side: those of sequence b start at place
// cu_q[b] / 32 + b, which leaves at most one place a sequence empty. (A grid over sequences and the longest one's chunks
// spent 1.57 ms on empty workgroups where two portions of 1000 tokens ran beside 250 decoded ones.) The products q k^T and k k^T do
// not depend on the head: the waves take a share of the key dimension each, and every wave then takes heads of the group.
// Step sizes: with room for two waves a SIMD asked for, the compiler keeps the accumulators beside the other registers and three fit: 70 -> 61 us
// (7 prompts of 2000 tokens on average, 32 heads of 128 x 64); four spill, 69.
template <typename T, int KIND, int D>
__global__ __launch_bounds__(256, KIND == kChunkDelta ? 4 : KIND == kChunkStep ? 2 : 1) void chunk_prep_kernel(ChunkParams p) {
  constexpr bool DELTA = KIND == kChunkDelta, SILU = KIND == kChunkConst;
  using Row4 = std::conditional_t<sizeof(T) == 2, uint2, float4>;      // four entries as they lie in memory
  auto wide = [](Row4 x) __attribute__((always_inline)) { return ld4(reinterpret_cast<const T*>(&x)); };
  constexpr int RS = kCh + 1;
  __shared__ float prod[4][kCh * RS];                  // partial products of the waves
  __shared__ __attribute__((aligned(16))) float amat[DELTA ? 4 : 1][kCh * (kCh + kPad)];
  __shared__ float powers[KIND == kChunkConst ? 4 : 1][kCh + 1];
  const int g = blockIdx.y, place = blockIdx.x, cu0 = p.cu_q[0];
  int b = -1;
  for (int i0 = 0; i0 < p.B; i0 += kWave) {            // the last sequence that starts at this place or before
    const int i = i0 + (threadIdx.x & 63);
    const uint64_t starts = __builtin_amdgcn_ballot_w64(i < p.B && (p.cu_q[min(i, p.B)] - cu0) / kCh + i <= place);
    b += __builtin_popcountll(starts);
    if (starts != ~0ull) break;
  }
  const int q0 = p.cu_q[b], n = p.cu_q[b + 1] - q0;
  const int c0 = (place - (q0 - cu0) / kCh - b) * kCh;
  if (c0 >= n) return;
  const int cn = min(kCh, n - c0);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, half = lane >> 5;
  const int64_t t0 = static_cast<int64_t>(q0) + c0;
  const int rep = p.H / p.G;
  // what the first head's decays are made of, requested with the rows
  float first_a = 0.0f, first_g = 0.0f;
  T first_step{};
  if (KIND != kChunkConst && w < rep && r < cn) {
    const int64_t at = (t0 + r) * p.H + g * rep + w;
    if constexpr (KIND == kChunkStep) first_step = static_cast<const T*>(p.a)[(t0 + r) * p.lda + g * rep + w];
    if constexpr (DELTA) {
      first_a = static_cast<const float*>(p.a)[at];
      first_g = p.decay[at];
    }
  }
  {
    const bool kk = DELTA && w < 2;                    // delta rule: waves 0, 1 k k^T, waves 2, 3 q k^T; otherwise all q k^T
    constexpr int shares = DELTA ? 2 : 4;
    const int r_in = min(r, cn - 1);                   // tokens past the end: the last one's rows, not used
    const int share = DELTA ? (w & 1) : w;
    const T* left = static_cast<const T*>(kk ? p.k : p.q) + (t0 + r_in) * (kk ? p.ldk : p.ldq) + static_cast<int64_t>(g) * D;
    const T* right = static_cast<const T*>(p.k) + (t0 + r_in) * p.ldk + static_cast<int64_t>(g) * D;
    if (DELTA && !kk) {
      // q k^T in 64 bits: read-outs are sums of few of these products, each a small difference of large terms. Summed in f32 they
      // were most of an output's error (1.33e-7 at heads of 128 x 128; 0.86e-7 with these, 0.95e-7 in the token loop).
      const int r16 = lane & 15, quad = lane >> 4;
      f64x4 acc[2][2];
#pragma unroll
      for (int x = 0; x < 4; ++x) acc[x >> 1][x & 1] = f64x4{0.0, 0.0, 0.0, 0.0};
      const T* q16 = static_cast<const T*>(p.q) + t0 * p.ldq + static_cast<int64_t>(g) * D + 4 * quad;
      const T* k16 = static_cast<const T*>(p.k) + t0 * p.ldk + static_cast<int64_t>(g) * D + 4 * quad;
      Row4 x[D / 32][2], y[D / 32][2];                 // all of them on their way at once
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int64_t row = min(16 * e + r16, cn - 1);
          x[i][e] = *reinterpret_cast<const Row4*>(q16 + row * p.ldq + share * 16 + 32 * i);
          y[i][e] = *reinterpret_cast<const Row4*>(k16 + row * p.ldk + share * 16 + 32 * i);
        }
#pragma unroll
      for (int i = 0; i < D / 32; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f64x4& to = acc[e >> 1][e & 1];
          const float4 none{0.0f, 0.0f, 0.0f, 0.0f};
          const float4 a = 16 * (e >> 1) + r16 < cn ? wide(x[i][e >> 1]) : none, b = 16 * (e & 1) + r16 < cn ? wide(y[i][e & 1]) : none;
          to = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, to, 0, 0, 0);
          to = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.y, to, 0, 0, 0);
          to = __builtin_amdgcn_mfma_f64_16x16x4f64(a.z, b.z, to, 0, 0, 0);
          to = __builtin_amdgcn_mfma_f64_16x16x4f64(a.w, b.w, to, 0, 0, 0);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)                      // (its result rows are lane / 16 + 4 i)
#pragma unroll
        for (int i = 0; i < 4; ++i) prod[w][(16 * (e >> 1) + quad + 4 * i) * RS + 16 * (e & 1) + r16] = static_cast<float>(acc[e >> 1][e & 1][i]);
    } else {
      const bool in = r < cn;
      f32x16 acc, acc2;                                  // two sums of half the length: half the roundings each
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = acc2[i] = 0.0f;
      constexpr int N = D / (8 * shares);
      Row4 xr[N], yr[N];                               // all of them on their way at once
#pragma unroll
      for (int i = 0; i < N; ++i) {
        xr[i] = *reinterpret_cast<const Row4*>(left + (share + i * shares) * 8 + 4 * half);
        yr[i] = *reinterpret_cast<const Row4*>(right + (share + i * shares) * 8 + 4 * half);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const float4 none{0.0f, 0.0f, 0.0f, 0.0f};
        const float4 x = in ? chunk_act<SILU>(wide(xr[i])) : none, y = in ? chunk_act<SILU>(wide(yr[i])) : none;
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, y.x, acc, 0, 0, 0);
        acc2 = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, y.y, acc2, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.z, y.z, acc, 0, 0, 0);
        acc2 = __builtin_amdgcn_mfma_f32_32x32x2f32(x.w, y.w, acc2, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) prod[w][acc_row(i, half) * RS + r] = acc[i] + acc2[i];
    }
  }
  __syncthreads();
  const uint32_t p_off = static_cast<uint32_t>(4 * half * p.H * kCh) + r;
  int r_here = r, half_here = half, cn_here = cn;
#pragma unroll 1
  for (int hr = w; hr < rep; hr += 4) {
    asm volatile("" : "+v"(r_here), "+v"(half_here), "+s"(cn_here) : : "memory");      // masks and reads stay in the loop: hoisted they spill
    const int r = r_here, half = half_here, cn = cn_here;
    const int h = g * rep + hr;
    // lane = token (both halves alike): decay, factor of the written value
    float dec = 1.0f, wr = 1.0f;
    if (r < cn) {
      const int64_t at = (t0 + r) * p.H + h;
      if constexpr (KIND == kChunkStep) {
        const T step = hr == w ? first_step : static_cast<const T*>(p.a)[(t0 + r) * p.lda + h];
        wr = softplusf_(ldf(&step) + p.p0[h]);
        dec = expf(-expf(p.p1[h]) * wr);
      } else if constexpr (DELTA) {
        wr = hr == w ? first_a : static_cast<const float*>(p.a)[at];       // beta
        dec = hr == w ? first_g : p.decay[at];
      }
    } else {
      wr = 0.0f;
    }
    // G_t and E_t w_t, lane = t; D_tj w_j, lane = j with t in the result layout's registers (w = 1 but for step sizes). The products
    // are formed in 64 bits and rounded once: a constant decay rounds the same way at every step, and its error would grow with the
    // tokens it spans.
    float gt = 1.0f, et = 1.0f;
    float dm[16];
    if constexpr (KIND == kChunkConst) {
      double pw = 1.0, sq = p.decay[h];
      for (int e = lane; e > 0; e >>= 1, sq *= sq)
        if (e & 1) pw *= sq;
      if (lane <= kCh) powers[w][lane] = static_cast<float>(pw);
      __builtin_amdgcn_wave_barrier();
      gt = powers[w][r + 1];
      et = powers[w][max(cn - 1 - r, 0)];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int e = acc_row(i, half) - r;
        dm[i] = e >= 0 ? powers[w][max(e, 0)] : 0.0f;
      }
      __builtin_amdgcn_wave_barrier();
    } else {
      double run = 1.0, back = 1.0, col = 0.0;
#pragma unroll
      for (int t = 0; t < kCh; ++t) {
        const double gd = chunk_lane(dec, t);
        run *= gd;
        gt = r == t ? static_cast<float>(run) : gt;
        col = r == t ? (DELTA ? 1.0 : static_cast<double>(wr)) : col * gd;       // zero above the diagonal
        const float colf = static_cast<float>(col);
        if (((t >> 2) & 1) == 0) dm[4 * (t >> 3) + (t & 3)] = colf;   // rows of the lower half of the lanes
        else dm[4 * (t >> 3) + (t & 3)] = half ? colf : dm[4 * (t >> 3) + (t & 3)];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = kCh - 1; t >= 0; --t) {
        et = r == t ? static_cast<float>(back * (DELTA ? 1.0 : static_cast<double>(wr))) : et;
        back *= chunk_lane(dec, t);
      }
    }
    if (half == 0 && r < cn) {
      p.Gf[(t0 + r) * p.H + h] = gt;
      p.Ef[(t0 + r) * p.H + h] = et;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = acc_row(i, half);
      float x;
      if constexpr (DELTA) x = prod[2][t * RS + r] + prod[3][t * RS + r];
      else x = (prod[0][t * RS + r] + prod[1][t * RS + r]) + (prod[2][t * RS + r] + prod[3][t * RS + r]);
      x *= dm[i];
      x = r <= t ? x : 0.0f;                           // selected: what a later token brings may not be finite
      if (t < cn) p.P[((t0 + 8 * (i >> 2) + (i & 3)) * p.H + h) * kCh + p_off] = x;
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (DELTA) {
      constexpr int AS = kCh + kPad;
      float* am = amat[w];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int t = acc_row(i, half);
        const float x = prod[0][t * RS + r] + prod[1][t * RS + r];
        // lanes hold beta of token r: the row's own beta is another lane's
        am[t * AS + r] = r < t ? x * dm[i] : 0.0f;
      }
      __builtin_amdgcn_wave_barrier();
      // column r of (I + diag(beta) A)^-1 by forward substitution, times beta_r (the row of diag(beta) on the right)
      float x[kCh];
#pragma unroll
      for (int t = 0; t < kCh; ++t) {
        float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < t; i += 4) {
          const float4 av = *reinterpret_cast<const float4*>(am + t * AS + i);
          s[0] += av.x * x[i];
          if (i + 1 < t) s[1] += av.y * x[i + 1];
          if (i + 2 < t) s[2] += av.z * x[i + 2];
          if (i + 3 < t) s[3] += av.w * x[i + 3];
        }
        x[t] = (r == t ? 1.0f : 0.0f) - chunk_lane(wr, t) * ((s[0] + s[1]) + (s[2] + s[3]));
        asm volatile("" : "+v"(x[t]) : : "memory");    // a row's reads at a time: hoisted ones spill
      }
#pragma unroll
      for (int t = 0; t < kCh; ++t)
        if (t < cn && (t & 1) == half) p.Tm[((t0 + t) * p.H + h) * kCh + r] = r <= t ? x[t] * wr : 0.0f;
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// Three bf16 numbers whose sum is a finite f32 value: its 24 bits cut into eights, so that nothing is rounded. As operands of the bf16
// matrix instructions (exact products, f32 sums) they give f32 products at four to eight times the f32 instructions' rate. An
// infinity has no such pieces: a wave that meets one computes its chunk on the f32 instructions.
struct Pieces4 { uint2 p[3]; };
__device__ __forceinline__ uint32_t high_halves(float a, float b) {
  return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302u);
}
__device__ __forceinline__ float below_high(float a) { return a - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, a) & 0xffff0000u); }
__device__ __forceinline__ Pieces4 cut4(float x, float y, float z, float w) {
  Pieces4 r;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    r.p[i] = uint2{high_halves(x, y), high_halves(z, w)};
    if (i < 2) { x = below_high(x); y = below_high(y); z = below_high(z); w = below_high(w); }
  }
  return r;
}
__device__ __forceinline__ chunk_bf16x8 join8(uint2 lo, uint2 hi) {
  return __builtin_bit_cast(chunk_bf16x8, uint4{lo.x, lo.y, hi.x, hi.y});
}

// MODE 0: the whole sequence; 1: what a segment adds to the state, and its decay; 2: a segment from its starting state.
// grid: (heads / HPW * column parts, segments, sequences), NW waves on 16 columns of the state each: the columns of one head,
// or of HPW heads of one group (they share q and k). Sixteen columns and not 32: a compute unit that gets one workgroup then
// holds two waves a SIMD, and one's LDS reads, staging and row factors run beside the other's products.
// NORM (delta rule, workgroups that hold whole heads): a chunk's outputs wait in registers for the barrier behind which the other waves' sums of
// squares are there, and leave normed and gated with the next chunk: no f32 rows through memory and no launch to read them back. 16 x 1024 tokens, 16
// heads of 128: 267 + 59 us in two launches, 307 in one (the layer 829 -> 814).
// CUT (delta rule, 128 rows of the state, eight waves): K^T U on the bf16 instructions, K and U cut into three pieces each (K once, where it is
// staged; the state's other products would have it cut in every chunk): 1024 clocks a wave and chunk for 2048 of the chain's 6900 at the f32 rate. Sixteen
// prompts of 1024 tokens, the layer 818 -> 803 us; 32 of 500 904 -> 888. States off 64 bits, pieces / f32 products: decays
// about 0.999, 1000 tokens, 1.6e-7 / 3.3e-7 (fewer roundings at the state's magnitude); fast decays, over all remainders of the last chunk, 6.8e-8 / 7.1e-8
// root mean square, 8.4 / 9.9 the largest (by the places of the last tokens in the sum 0.7 to 1.4 of the other's). Outputs 8.8e-8 either way there, 1.9e-7 / 3.1e-7. Constant decays gain nothing (833 / 836: their time is the silu of q, k and v), nor
// do launches of four waves (one prompt of 1000 250 / 255). Chunks with a value that is not finite take the f32 products.
template <typename T, int KIND, int DT, int NW, int HPW, int MODE, bool NORM = false, bool OWN = false>
__global__ __launch_bounds__(NW * 64, 2) void chunk_scan_kernel(ChunkParams p) {
  static_assert(!NORM || (KIND == kChunkDelta && MODE == 0), "the norm follows the delta rule's whole sequences");
  static_assert(!OWN || KIND == kChunkConst, "the other decays are the tokens' own");
  constexpr bool DELTA = KIND == kChunkDelta, SILU = KIND == kChunkConst, FULL = MODE != 1;
  constexpr int D = DT * 16, RS = D + kPad, PS = kCh + kPad, NT = NW * 64, WPW = NW / HPW;
  constexpr int SLOTS = OWN ? 3 : 2, RAW = 20;                 // RAW: floats of a row of q k^T
  constexpr int MATS = FULL && !OWN ? HPW * (DELTA ? 2 : 1) : 0;       // P of every head, then T of every head
  constexpr bool CUT = DELTA && DT == 8 && NW == 8;            // K^T U from pieces
  constexpr int KB = D * 2 + 16, kImg = kCh * KB;              // bytes of a row and of an image of pieces
  __shared__ __attribute__((aligned(16))) unsigned char kc_all[2][CUT ? 3 * kImg : 16];
  __shared__ int odd_all[2][NW];                               // whether a wave staged a k that is not finite
  __shared__ __attribute__((aligned(16))) float k_all[SLOTS][kCh * RS];
  __shared__ __attribute__((aligned(16))) float q_all[SLOTS][FULL ? kCh * RS : 4];
  __shared__ __attribute__((aligned(16))) float raw_all[2][OWN && FULL ? 8 * 16 * RAW : 4], pw_all[OWN ? NW : 1][OWN ? kCh + 4 : 4];
  __shared__ __attribute__((aligned(16))) float pt_all[2][MATS > 0 ? MATS : 1][MATS > 0 ? kCh * PS : 4];
  __shared__ __attribute__((aligned(16))) float ge_all[2][HPW][OWN ? 4 : 2 * kCh];      // G, then E
  __shared__ __attribute__((aligned(16))) float sq_all[2][NORM ? NW : 1][NORM ? kCh : 4], inv_all[NORM ? NW : 1][NORM ? kCh : 4];
  const int b = blockIdx.z;
  const int q0 = p.cu_q[b], n_all = p.cu_q[b + 1] - q0;
  const int s0 = MODE == 0 ? 0 : blockIdx.y * p.seg_len;
  const int s1 = MODE == 0 ? n_all : min(n_all, s0 + p.seg_len);
  if (s0 >= n_all || (MODE == 1 && s1 == n_all)) return;       // what the last segment adds is nobody's start
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, quad = lane >> 4;
  const int parts = p.Dv / 16 / WPW;                           // 1 where several heads share the workgroup
  const int h0 = static_cast<int>(blockIdx.x) / parts * HPW, hw = w / WPW, h = h0 + hw;         // (uniform over a wave)
  const int col = ((static_cast<int>(blockIdx.x) % parts) * WPW + w % WPW) * 16 + r;
  const int g = h0 / (p.H / p.G);
  const T* kp = static_cast<const T*>(p.k) + static_cast<int64_t>(q0) * p.ldk + static_cast<int64_t>(g) * D;
  const T* qp = static_cast<const T*>(p.q) + static_cast<int64_t>(q0) * p.ldq + static_cast<int64_t>(g) * D;
  const T* vp = static_cast<const T*>(p.v) + static_cast<int64_t>(q0) * p.ldv + static_cast<int64_t>(h) * p.Dv;
  const int64_t row0 = static_cast<int64_t>(q0) * p.H;
  float* sbase = p.state + (static_cast<int64_t>(p.slots[b]) * p.H + h) * D * p.Dv;
  float* gbase = MODE == 0 ? nullptr : p.seg_state + ((static_cast<int64_t>(b) * p.segs + blockIdx.y) * p.H + h) * D * p.Dv;

  // addresses are a uniform row plus a lane's 32-bit offset inside it
  const uint32_t st_off = static_cast<uint32_t>(4 * quad * p.Dv) + col;
  f32x4 S[DT];
  {
    const bool carry = MODE == 2 ? p.segs > 0 : MODE == 0 && p.ctx_lens[b] > 0;
    const float* from = MODE == 2 ? gbase : sbase;
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[j][i] = carry ? from[(16 * j + i) * p.Dv + st_off] : 0.0f;
  }
  float skip = 0.0f;
  if (KIND == kChunkStep && FULL) skip = p.p2[h];
  // a whole chunk's decay in two parts: a constant one, rounded, would be off the same way in every chunk
  double g_chunk = 1.0, seg_dec = 1.0;
  float g_rest = 0.0f;
  if constexpr (KIND == kChunkConst) {
    g_chunk = p.decay[h];
#pragma unroll
    for (int i = 1; i < kCh; i *= 2) g_chunk *= g_chunk;
    g_rest = static_cast<float>(g_chunk - static_cast<double>(static_cast<float>(g_chunk)));
  }
  // constant decays: their powers, formed in 64 bits and rounded once; G and E of a whole chunk, and D of this lane's entries of P
  float4 g_fac[2], e_fac[2];
  float d_diag[4], d_low[4];
  if constexpr (OWN) {
    double pw = 1.0, sq = p.decay[h];
    for (int e = lane; e > 0; e >>= 1, sq *= sq)
      if (e & 1) pw *= sq;
    if (lane <= kCh) pw_all[w][lane] = static_cast<float>(pw);
    __builtin_amdgcn_wave_barrier();                   // (a wave's LDS operations keep their order)
    const float* of = pw_all[w];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int t = 16 * x + 4 * quad;
      g_fac[x] = float4{of[t + 1], of[t + 2], of[t + 3], of[t + 4]};
      e_fac[x] = float4{of[31 - t], of[30 - t], of[29 - t], of[28 - t]};
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      d_diag[i] = of[max(r - 4 * quad - i, 0)];
      d_low[i] = of[16 + r - 4 * quad - i];
    }
  }

  // the next chunk's rows on their way, as they lie in memory (a conversion here would wait for them): q and k four entries a thread, P
  // and T too, a value for each of the wave's 32 x 16
  constexpr int KQ = kCh * D / 4 / NT, PN = (MATS * kCh * kCh / 4 + NT - 1) / NT, PX = PN > 0 ? PN : 1;
  static_assert(kCh * D / 4 % NT == 0, "whole rows of q and k a step");
  using Row4 = std::conditional_t<SILU, uint2, float4>;
  using Entry = std::conditional_t<SILU, uint32_t, float>;
  Row4 kreg[KQ], qreg[FULL ? KQ : 1];
  float4 preg[PX];
  Entry vreg[8];
  float gereg;
  const uint32_t kq_off = static_cast<uint32_t>(threadIdx.x % (D / 4) * 4);
  const int kq_tok = threadIdx.x / (D / 4);
  const uint32_t k_off = kq_tok * static_cast<uint32_t>(p.ldk) + kq_off, q_off = kq_tok * static_cast<uint32_t>(p.ldq) + kq_off;
  const uint32_t v_off = 4 * quad * static_cast<uint32_t>(p.ldv) + col;
  const uint32_t o_off = static_cast<uint32_t>(4 * quad * p.H * p.Dv) + col;
  const uint32_t ge_off = static_cast<uint32_t>((lane & 31) * p.H + hw);
  const int p_tok = (threadIdx.x >> 3) & 31;
  const uint32_t p_off = static_cast<uint32_t>(p_tok * p.H * kCh + (threadIdx.x & 7) * 4);
  auto entry = [](const T* at) __attribute__((always_inline)) {
    if constexpr (SILU) return static_cast<uint32_t>(at->bits);
    else return *at;
  };
  auto four = [](Row4 x) __attribute__((always_inline)) {
    if constexpr (SILU) return chunk_act<true>(ld4(reinterpret_cast<const bf16_t*>(&x)));
    else return x;
  };
  // parts of a chunk: k and q, and what else it needs (one function by parts, not two: where both go together the compiler orders their loads and
  // the products otherwise, delta rule of 64 x 128, 16 heads in 4 groups, 16 of 290 to 1680 tokens 341 us for 327)
  using Both = std::integral_constant<int, 3>;
  using KeysQueries = std::integral_constant<int, 1>;
  using Rest = std::integral_constant<int, 2>;
  auto fetch_rows = [&](int c0, auto whole, auto part) __attribute__((always_inline)) {
    constexpr bool WHOLE = decltype(whole)::value;     // all 32 tokens are there: loads without conditions
    constexpr int PART = decltype(part)::value;
    const int cn = s1 - c0;
#pragma unroll
    for (int it = 0; it < (PART & 1 ? KQ : 0); ++it) {
      constexpr int per = NT / (D / 4);
      const bool in = WHOLE || kq_tok + it * per < cn;
      kreg[it] = in ? *reinterpret_cast<const Row4*>(kp + static_cast<int64_t>(c0 + it * per) * p.ldk + k_off) : Row4{};
      if constexpr (FULL) qreg[it] = in ? *reinterpret_cast<const Row4*>(qp + static_cast<int64_t>(c0 + it * per) * p.ldq + q_off) : Row4{};
    }
    if constexpr (!(PART & 2)) return;
#pragma unroll
    for (int it = 0; it < PN; ++it) {
      const int m = (it * NT + (w << 6)) >> 8;         // matrix of this wave's pieces
      const bool in = m < MATS && (WHOLE || p_tok < cn);
      const float* from = DELTA && m >= HPW ? p.Tm : p.P;
      const int64_t at = (row0 + static_cast<int64_t>(c0) * p.H + h0 + (DELTA && m >= HPW ? m - HPW : m)) * kCh;
      preg[it] = in ? ld4(from + at + p_off) : float4{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int lo = 16 * (i >> 2) + (i & 3);
      vreg[i] = WHOLE || lo + 4 * quad < cn ? entry(vp + static_cast<int64_t>(c0 + lo) * p.ldv + v_off) : Entry{};
    }
    if constexpr (OWN) return;
    const bool in = WHOLE || (lane & 31) < cn;         // lane = token, G in the lower half of the lanes, E in the upper
    const int64_t at = row0 + static_cast<int64_t>(c0) * p.H + h0;
    gereg = in ? (lane >= 32 ? p.Ef : p.Gf)[at + ge_off] : 0.0f;
  };
  auto fetch = [&](int c0, auto part) __attribute__((always_inline)) {
    if (s1 - c0 >= kCh) fetch_rows(c0, std::true_type{}, part);
    else fetch_rows(c0, std::false_type{}, part);
  };
  // rows 16 x + 4 quad .. + 3 of a vector, a row of a left-hand matrix from column 16 j on
  auto rows4 = [&](const float* from, int x) __attribute__((always_inline)) {
    return *reinterpret_cast<const float4*>(from + 16 * x + 4 * quad);
  };
  auto left = [&](const float* m, int stride, int x, int j) __attribute__((always_inline)) {
    return *reinterpret_cast<const float4*>(m + (16 * x + r) * stride + 16 * j + 4 * quad);
  };
  auto mul4 = [&](f32x4 acc, float4 a, f32x4 bb) __attribute__((always_inline)) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, bb[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, bb[1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, bb[2], acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, bb[3], acc, 0, 0, 0);
  };
  auto scale4 = [&](f32x4 x, float4 f) __attribute__((always_inline)) { return f32x4{x[0] * f.x, x[1] * f.y, x[2] * f.z, x[3] * f.w}; };
  const f32x4 zero{0.0f, 0.0f, 0.0f, 0.0f};
  // y += m x for a lower triangular m. The products run over whole 16 x 16 blocks, in which a token's value meets the zeros of the
  // tokens before it: one that is not finite would reach them, so a wave that sees one goes token by token.
  auto triangle = [&](f32x4 (&y)[2], const float* m, const f32x4 (&x)[2]) __attribute__((always_inline)) {
    float z = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) z = fmaf(x[i >> 2][i & 3], 0.0f, z);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(z != 0.0f) == 0, 1)) {
      y[0] += mul4(zero, left(m, PS, 0, 0), x[0]);
      y[1] += mul4(mul4(zero, left(m, PS, 1, 0), x[0]), left(m, PS, 1, 1), x[1]);
      return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll 1
      for (int from = 0; from < 4; ++from) {
        const int j = 16 * (i >> 2) + 4 * from + (i & 3);
        const float v = __shfl(x[i >> 2][i & 3], 16 * from + r, kWave);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int t = 16 * (k >> 2) + 4 * quad + (k & 3);
          y[k >> 2][k & 3] = j <= t ? fmaf(m[t * PS + j], v, y[k >> 2][k & 3]) : y[k >> 2][k & 3];
        }
      }
  };
  // NORM: the chunk before, its gates, and what is left to do for it
  f32x4 done[2] = {zero, zero};
  uint32_t gates[8];
  const float col_w = NORM ? p.norm_w[col] : 0.0f;
  const uint32_t gate_off = NORM ? static_cast<uint32_t>(4 * quad) * static_cast<uint32_t>(p.ld_gate) + h * p.Dv + col : 0u;
  auto finish = [&](int buf, int c0, int cn) __attribute__((always_inline)) {
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < WPW; ++i) ss += sq_all[buf][hw * WPW + i][lane & 31];
    inv_all[w][lane & 31] = 1.0f / sqrtf(ss / static_cast<float>(p.Dv) + p.eps);      // (a wave's LDS operations keep their order)
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const float4 inv = rows4(inv_all[w], x);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float gv = __builtin_bit_cast(float, gates[4 * x + i] << 16), f = i == 0 ? inv.x : i == 1 ? inv.y : i == 2 ? inv.z : inv.w;
        const float y = done[x][i] * f * col_w * (p.gate_silu ? quick_silu_(gv) : sigmoidf_(gv));
        const int lo = 16 * x + i;
        if (lo + 4 * quad < cn) stf(reinterpret_cast<bf16_t*>(p.o) + (row0 + static_cast<int64_t>(c0 + lo) * p.H + h) * p.Dv + o_off, y);
      }
    }
  };
  f32x4 U_next[2];
  auto stage = [&](int buf, auto part) __attribute__((always_inline)) {
    constexpr int PART = decltype(part)::value;
    float odd_k = 0.0f;                                // NaN if a value is not finite
#pragma unroll
    for (int it = 0; it < (PART & 1 ? KQ : 0); ++it) {
      const int tok = kq_tok + it * (NT / (D / 4)), at = tok * RS + kq_off;
      const float4 kv = four(kreg[it]);
      st4(k_all[buf] + at, kv);
      if constexpr (CUT) {
        odd_k = fmaf(kv.x, 0.0f, fmaf(kv.y, 0.0f, fmaf(kv.z, 0.0f, fmaf(kv.w, 0.0f, odd_k))));
        const Pieces4 c = cut4(kv.x, kv.y, kv.z, kv.w);
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<uint2*>(kc_all[buf] + i * kImg + tok * KB + 2 * kq_off) = c.p[i];
      }
      if constexpr (FULL) st4(q_all[buf] + at, four(qreg[it]));
    }
    if constexpr (CUT) {
      const bool odd = __builtin_amdgcn_ballot_w64(odd_k != 0.0f) != 0;
      if (lane == 0) odd_all[buf][w] = odd;
    }
    if constexpr (!(PART & 2)) return;
#pragma unroll
    for (int it = 0; it < PN; ++it) {
      const int m = (it * NT + (w << 6)) >> 8;
      if (m < MATS) st4(pt_all[buf][m] + p_tok * PS + (threadIdx.x & 7) * 4, preg[it]);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if constexpr (SILU) U_next[i >> 2][i & 3] = quick_silu_(__builtin_bit_cast(float, vreg[i] << 16));
      else U_next[i >> 2][i & 3] = vreg[i];
    }
    if (!OWN && w % WPW == 0) ge_all[buf][hw][lane] = gereg;
  };
  // OWN: parts of q k^T, which does not depend on the head, of the chunk in a slot: the waves' shares of the blocks (0, 0), (1, 1) by halves of the
  // key dimension and of (1, 0) by quarters. A lane gets four keys of its query: entries as `left` reads them.
  auto raw_parts = [&](int slot, float* to) __attribute__((always_inline)) {
    auto part = [&](int number, int xq, int xk, int from, auto count) __attribute__((always_inline)) {
      constexpr int N = decltype(count)::value;
      constexpr int M = DT == 4 ? 2 * N : N;           // sums of 16 products, of eight at 64 rows
      f32x4 sum[M];
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const float4 qv = left(q_all[slot], RS, xq, from + j), kv = left(k_all[slot], RS, xk, from + j);
        sum[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.x, qv.x, zero, 0, 0, 0);
        sum[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.y, qv.y, sum[j], 0, 0, 0);
        f32x4& rest = sum[M - N + j];
        rest = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.z, qv.z, M > N ? zero : rest, 0, 0, 0);
        rest = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.w, qv.w, rest, 0, 0, 0);
      }
#pragma unroll
      for (int o = M / 2; o > 0; o /= 2)
#pragma unroll
        for (int j = 0; j < o; ++j) sum[j] += sum[j + o];
      *reinterpret_cast<f32x4*>(to + (number * 16 + r) * RAW + 4 * quad) = sum[0];
    };
    const int a = w & 3;
    if (NW == 4 || w < 4) part(a, a >> 1, a >> 1, (a & 1) * (DT / 2), std::integral_constant<int, DT / 2>{});
    if (NW == 4 || w >= 4) part(4 + a, 1, 0, a * (DT / 4), std::integral_constant<int, DT / 4>{});
  };
  auto raw4 = [&](const float* raw, int number) __attribute__((always_inline)) { return ld4(raw + (number * 16 + r) * RAW + 4 * quad); };
  auto add4 = [](float4 a, float4 b) __attribute__((always_inline)) { return float4{a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w}; };
  // y += P x with P = D o q k^T (compare triangle)
  auto own_triangle = [&](f32x4 (&y)[2], const float* raw, const f32x4 (&x)[2]) __attribute__((always_inline)) {
    float z = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) z = fmaf(x[i >> 2][i & 3], 0.0f, z);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(z != 0.0f) == 0, 1)) {
      auto diagonal = [&](int number) __attribute__((always_inline)) {
        const float4 a = add4(raw4(raw, number), raw4(raw, number + 1));
        const int e = r - 4 * quad;                    // selected: what a later token brings may not be finite
        return float4{e >= 0 ? a.x * d_diag[0] : 0.0f, e >= 1 ? a.y * d_diag[1] : 0.0f, e >= 2 ? a.z * d_diag[2] : 0.0f, e >= 3 ? a.w * d_diag[3] : 0.0f};
      };
      const float4 a = add4(add4(raw4(raw, 4), raw4(raw, 5)), add4(raw4(raw, 6), raw4(raw, 7)));
      const float4 low{a.x * d_low[0], a.y * d_low[1], a.z * d_low[2], a.w * d_low[3]};
      y[0] += mul4(zero, diagonal(0), x[0]);
      y[1] += mul4(mul4(zero, low, x[0]), diagonal(2), x[1]);
      return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll 1
      for (int from = 0; from < 4; ++from) {
        const int j = 16 * (i >> 2) + 4 * from + (i & 3);
        const float v = __shfl(x[i >> 2][i & 3], 16 * from + r, kWave);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int t = 16 * (k >> 2) + 4 * quad + (k & 3);
          const float* at = raw + (t & 15) * RAW + (j & 15);
          constexpr int next = 16 * RAW;
          const float m = (t >> 4) == (j >> 4) ? at[2 * (t >> 4) * next] + at[(2 * (t >> 4) + 1) * next]
                                               : (at[4 * next] + at[5 * next]) + (at[6 * next] + at[7 * next]);
          y[k >> 2][k & 3] = j <= t ? fmaf(m * pw_all[w][max(t - j, 0)], v, y[k >> 2][k & 3]) : y[k >> 2][k & 3];
        }
      }
  };
  // Two buffers: a chunk is staged while the one before it is computed, each wave at its own time, and two chunks ahead are on
  // their way in registers. One barrier a chunk. OWN: three of k and q, staged a chunk earlier, since q k^T of a chunk is formed during the one before.
  int slot = 0;
  if constexpr (OWN) {
    auto rows = [&](int c0) __attribute__((always_inline)) {
      if (c0 < s1) fetch(c0, KeysQueries{});
    };
    rows(s0);
    stage(0, KeysQueries{});
    rows(s0 + kCh);
    stage(1, KeysQueries{});
    rows(s0 + 2 * kCh);
    fetch(s0, Rest{});
    stage(0, Rest{});
    if (s0 + kCh < s1) fetch(s0 + kCh, Rest{});
    __syncthreads();
    if constexpr (FULL) raw_parts(0, raw_all[0]);
  } else {
    fetch(s0, Both{});
    stage(0, Both{});
    if (s0 + kCh < s1) fetch(s0 + kCh, Both{});
  }
  __syncthreads();
  int buf = 0;
  for (int c0 = s0; c0 < s1; c0 += kCh, buf ^= 1) {
    const int cn = min(kCh, s1 - c0);
    const int here = OWN ? slot : buf, next_slot = here == 2 ? 0 : here + 1, last_slot = here == 0 ? 2 : here - 1;
    const float *k_lds = k_all[here], *q_lds = q_all[here];
    const auto& pt_lds = pt_all[buf];
    const auto& ge_lds = ge_all[buf];
    if constexpr (NORM) {
      if (c0 > s0) finish(buf ^ 1, c0 - kCh, kCh);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int lo = 16 * (i >> 2) + (i & 3);
        gates[i] = lo + 4 * quad < cn ? p.gate[(static_cast<int64_t>(q0) + c0 + lo) * p.ld_gate + gate_off].bits : 0u;
      }
    }
    f32x4 U[2] = {U_next[0], U_next[1]};
    f32x4 o[2], u2[2];
    if constexpr (FULL) {
      f32x4 ks[2][2], qs[4][2];                        // [sum][rows]: several sums each, shorter and with fewer roundings
#pragma unroll
      for (int x = 0; x < 2; ++x) qs[0][x] = qs[1][x] = qs[2][x] = qs[3][x] = ks[0][x] = ks[1][x] = zero;
#pragma unroll
      for (int j = 0; j < DT; ++j) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          if constexpr (DELTA) ks[j & 1][x] = mul4(ks[j & 1][x], left(k_lds, RS, x, j), S[j]);
          qs[j & 3][x] = mul4(qs[j & 3][x], left(q_lds, RS, x, j), S[j]);
        }
      }
      if constexpr (DELTA) {
        f32x4 rest[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) rest[x] = U[x] - scale4(ks[0][x] + ks[1][x], rows4(ge_lds[hw], x));
        U[0] = U[1] = zero;
        triangle(U, pt_lds[HPW + hw], rest);
      }
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        o[x] = scale4((qs[0][x] + qs[1][x]) + (qs[2][x] + qs[3][x]), OWN ? g_fac[x] : rows4(ge_lds[hw], x));
        if constexpr (KIND == kChunkStep) o[x] += skip * U[x];
      }
      if constexpr (OWN) own_triangle(o, raw_all[buf], U);
      else triangle(o, pt_lds[hw], U);
    }
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      if constexpr (OWN) {
        float4 e = e_fac[x];
        if (cn < kCh) {                                // (tokens past the end are zeros)
          const int at = cn - 1 - 16 * x - 4 * quad;
          e = float4{pw_all[w][max(at, 0)], pw_all[w][max(at - 1, 0)], pw_all[w][max(at - 2, 0)], pw_all[w][max(at - 3, 0)]};
        }
        u2[x] = scale4(U[x], e);
      } else {
        u2[x] = scale4(U[x], rows4(ge_lds[hw] + kCh, x));
      }
    }
    const float g_last = OWN ? pw_all[w][cn] : ge_lds[hw][cn - 1];
    bool odd = !CUT;
    if constexpr (CUT) {
      float z = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) z = fmaf(u2[i >> 2][i & 3], 0.0f, z);
      odd = __builtin_amdgcn_ballot_w64(z != 0.0f || odd_all[buf][lane & (NW - 1)] != 0) != 0;
    }
    if (CUT && __builtin_expect(!odd, 1)) {
      // lane slots of a product: tokens 4 quad .. + 3 and 16 + 4 quad .. + 3, as u2 has them; K^T comes transposed out of LDS
      using lds_bf16x4 = __attribute__((address_space(3))) chunk_bf16x4;
      const unsigned char* kt = kc_all[buf] + (4 * quad + (r >> 2)) * KB + 8 * (r & 3);
      const Pieces4 ua = cut4(u2[0][0], u2[0][1], u2[0][2], u2[0][3]), ub = cut4(u2[1][0], u2[1][1], u2[1][2], u2[1][3]);
      chunk_bf16x8 uc[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) uc[i] = join8(ua.p[i], ub.p[i]);
      stage(buf ^ 1, Both{});                          // (behind the last chunk for nobody: without a branch, among the products)
#pragma unroll
      for (int j = 0; j < DT; ++j) {
        chunk_bf16x8 kc[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const chunk_bf16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(kt + i * kImg + 32 * j));
          const chunk_bf16x4 c = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(kt + i * kImg + 16 * KB + 32 * j));
          kc[i] = chunk_bf16x8{a[0], a[1], a[2], a[3], c[0], c[1], c[2], c[3]};
        }
        f32x4 add = zero;
        auto mm = [&](int a, int c) __attribute__((always_inline)) { add = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kc[a], uc[c], add, 0, 0, 0); };
        mm(2, 1);                                      // smallest products first; the two least pieces' is below a rounding
        mm(1, 2);
        mm(2, 0);
        mm(0, 2);
        mm(1, 1);
        mm(1, 0);
        mm(0, 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) add[i] = fmaf(S[j][i], g_last, add[i]);
        mm(0, 0);
        S[j] = add;
      }
    } else {
      if constexpr (OWN) {
        stage(last_slot, KeysQueries{});
        if constexpr (FULL) raw_parts(next_slot, raw_all[buf ^ 1]);
        stage(0, Rest{});
      } else {
        stage(buf ^ 1, Both{});
      }
#pragma unroll
      for (int j = 0; j < DT; ++j) {
        // constant decays, slow as a rule: what the chunk adds in two sums of its own, for fewer roundings at the state's magnitude
        constexpr bool APART = KIND == kChunkConst;
        f32x4 add[2] = {APART ? zero : S[j] * g_last, zero};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          f32x4& to = add[APART ? i >> 2 : 0];
          to = __builtin_amdgcn_mfma_f32_16x16x4f32(k_lds[(16 * (i >> 2) + 4 * quad + (i & 3)) * RS + 16 * j + r], u2[i >> 2][i & 3], to, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          S[j][i] = APART ? fmaf(S[j][i], g_last, fmaf(S[j][i], cn == kCh ? g_rest : 0.0f, add[0][i] + add[1][i])) : add[0][i];
      }
    }
    if constexpr (OWN) {
      if (c0 + 3 * kCh < s1) fetch(c0 + 3 * kCh, KeysQueries{});
      if (c0 + 2 * kCh < s1) fetch(c0 + 2 * kCh, Rest{});
      slot = next_slot;
    } else if (c0 + 2 * kCh < s1) {
      fetch(c0 + 2 * kCh, Both{});
    }
    if constexpr (NORM) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        done[x] = o[x];
        const float4 ss{row16_sum(o[x][0] * o[x][0]), row16_sum(o[x][1] * o[x][1]), row16_sum(o[x][2] * o[x][2]), row16_sum(o[x][3] * o[x][3])};
        if (r == 0) st4(&sq_all[buf][w][16 * x + 4 * quad], ss);
      }
    } else if constexpr (FULL) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int lo = 16 * (i >> 2) + (i & 3);
        if (lo + 4 * quad < cn) p.o[(row0 + static_cast<int64_t>(c0 + lo) * p.H + h) * p.Dv + o_off] = o[i >> 2][i & 3];
      }
    }
    if constexpr (MODE == 1) seg_dec *= KIND == kChunkConst ? g_chunk : static_cast<double>(g_last);      // (only whole chunks)
    __syncthreads();                                   // the next chunk is complete, and nobody reads this one any more
  }
  if constexpr (NORM) {
    const int last = s1 - s0 - 1 & ~(kCh - 1);
    finish(buf ^ 1, s0 + last, s1 - s0 - last);
  }
  if (MODE == 1 || s1 == n_all) {
    float* to = MODE == 1 ? gbase : sbase;
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) to[(16 * j + i) * p.Dv + st_off] = S[j][i];
  }
  if (MODE == 1 && lane == 0) p.seg_decay[(static_cast<int64_t>(b) * p.segs + blockIdx.y) * p.H + h] = static_cast<float>(seg_dec);
}

// The same scan for step sizes, whose q, k and v rows are bf16: an f32 value on the other side of a product is cut into its pieces, and
// three products on the bf16 instructions (exact, summed in f32) do for an f32 one, at three sixteenths of its time. The state is cut
// anew in every chunk. A chunk's read-out, its addition to the state and the staging of the next one stand in one block of code, so that
// each one's products run beside the others' cutting and reads. us, f32 products -> this, with the kernel in front: 32 x 512 tokens, 32
// heads of 128 x 64, 273 -> 190; 16 x 512 of 64 x 64 98 -> 77; one of 4096 in segments of 256 121 -> 94. It stays far from the matrix
// rate (two waves a SIMD, some 3 us a chunk); more waves did not fit: at 128 registers it spills (315 us for the first).
// Against 64 bits outputs are 0.77e-7 off, 0.83e-7 before, states 0.53 to 0.69e-7, as before.
template <int DT, int NW, int HPW, int MODE>
__global__ __launch_bounds__(NW * 64, 2) void chunk_step_kernel(ChunkParams p) {
  constexpr bool FULL = MODE != 1;
  constexpr int D = DT * 16, RB = D * 2 + 16, PB = kCh * 2 + 16, NT = NW * 64, WPW = NW / HPW;      // RB, PB: bytes of an LDS row
  constexpr int MATS = FULL ? HPW : 0, kMatImg = kCh * PB;
  __shared__ __attribute__((aligned(16))) unsigned char k_all[2][kCh * RB];
  __shared__ __attribute__((aligned(16))) unsigned char q_all[2][FULL ? kCh * RB : 16];
  __shared__ __attribute__((aligned(16))) unsigned char p_all[2][MATS > 0 ? MATS : 1][MATS > 0 ? 3 * kMatImg : 16];
  __shared__ __attribute__((aligned(16))) float ge_all[2][HPW][2 * kCh];      // G, then E
  __shared__ int odd_all[2][NW];                       // whether a wave staged a q, k or P that is not finite
  const int b = blockIdx.z;
  const int q0 = p.cu_q[b], n_all = p.cu_q[b + 1] - q0;
  const int s0 = MODE == 0 ? 0 : blockIdx.y * p.seg_len;
  const int s1 = MODE == 0 ? n_all : min(n_all, s0 + p.seg_len);
  if (s0 >= n_all || (MODE == 1 && s1 == n_all)) return;       // what the last segment adds is nobody's start
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, quad = lane >> 4;
  const int parts = p.Dv / 16 / WPW;                           // 1 where several heads share the workgroup
  const int h0 = static_cast<int>(blockIdx.x) / parts * HPW, hw = w / WPW, h = h0 + hw;         // (uniform over a wave)
  const int col = ((static_cast<int>(blockIdx.x) % parts) * WPW + w % WPW) * 16 + r;
  const int g = h0 / (p.H / p.G);
  const uint16_t* kp = static_cast<const uint16_t*>(p.k) + static_cast<int64_t>(q0) * p.ldk + static_cast<int64_t>(g) * D;
  const uint16_t* qp = static_cast<const uint16_t*>(p.q) + static_cast<int64_t>(q0) * p.ldq + static_cast<int64_t>(g) * D;
  const uint16_t* vp = static_cast<const uint16_t*>(p.v) + static_cast<int64_t>(q0) * p.ldv + static_cast<int64_t>(h) * p.Dv;
  const int64_t row0 = static_cast<int64_t>(q0) * p.H;
  float* sbase = p.state + (static_cast<int64_t>(p.slots[b]) * p.H + h) * D * p.Dv;
  float* gbase = MODE == 0 ? nullptr : p.seg_state + ((static_cast<int64_t>(b) * p.segs + blockIdx.y) * p.H + h) * D * p.Dv;

  // addresses are a uniform row plus a lane's 32-bit offset inside it
  const uint32_t st_off = static_cast<uint32_t>(4 * quad * p.Dv) + col;
  f32x4 S[DT];
  {
    const bool carry = MODE == 2 ? p.segs > 0 : MODE == 0 && p.ctx_lens[b] > 0;
    const float* from = MODE == 2 ? gbase : sbase;
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[j][i] = carry ? from[(16 * j + i) * p.Dv + st_off] : 0.0f;
  }
  const float skip = FULL ? p.p2[h] : 0.0f;
  double seg_dec = 1.0;

  // the next chunk's rows on their way, as they lie in memory (a conversion here would wait for them): q and k four entries a thread, P
  // too, a value for each of the wave's 32 x 16
  constexpr int KQ = kCh * D / 4 / NT, PN = (MATS * kCh * kCh / 4 + NT - 1) / NT, PX = PN > 0 ? PN : 1;
  static_assert(kCh * D / 4 % NT == 0, "whole rows of q and k a step");
  uint2 kreg[KQ], qreg[FULL ? KQ : 1];
  float4 preg[PX];
  uint32_t vreg[8];
  float gereg;
  const int kq_d = threadIdx.x % (D / 4) * 4, kq_tok = threadIdx.x / (D / 4);
  const uint32_t k_off = kq_tok * static_cast<uint32_t>(p.ldk) + kq_d, q_off = kq_tok * static_cast<uint32_t>(p.ldq) + kq_d;
  const uint32_t v_off = 8 * quad * static_cast<uint32_t>(p.ldv) + col;
  const uint32_t o_off = static_cast<uint32_t>(8 * quad * p.H * p.Dv) + col;
  const uint32_t ge_off = static_cast<uint32_t>((lane & 31) * p.H + hw);
  const int p_tok = (threadIdx.x >> 3) & 31;
  const uint32_t p_off = static_cast<uint32_t>(p_tok * p.H * kCh + (threadIdx.x & 7) * 4);
  auto fetch_rows = [&](int c0, auto whole) __attribute__((always_inline)) {
    constexpr bool WHOLE = decltype(whole)::value;     // all 32 tokens are there: loads without conditions
    const int cn = s1 - c0;
#pragma unroll
    for (int it = 0; it < KQ; ++it) {
      constexpr int per = NT / (D / 4);
      const bool in = WHOLE || kq_tok + it * per < cn;
      kreg[it] = in ? *reinterpret_cast<const uint2*>(kp + static_cast<int64_t>(c0 + it * per) * p.ldk + k_off) : uint2{0, 0};
      if constexpr (FULL) qreg[it] = in ? *reinterpret_cast<const uint2*>(qp + static_cast<int64_t>(c0 + it * per) * p.ldq + q_off) : uint2{0, 0};
    }
#pragma unroll
    for (int it = 0; it < PN; ++it) {
      const int m = (it * NT + (w << 6)) >> 8;         // matrix of this wave's pieces
      const bool in = m < MATS && (WHOLE || p_tok < cn);
      preg[it] = in ? ld4(p.P + (row0 + static_cast<int64_t>(c0) * p.H + h0 + m) * kCh + p_off) : float4{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      vreg[i] = WHOLE || i + 8 * quad < cn ? vp[static_cast<int64_t>(c0 + i) * p.ldv + v_off] : 0u;
    const bool in = WHOLE || (lane & 31) < cn;         // lane = token, G in the lower half of the lanes, E in the upper
    const int64_t at = row0 + static_cast<int64_t>(c0) * p.H + h0;
    gereg = in ? (lane >= 32 ? p.Ef : p.Gf)[at + ge_off] : 0.0f;
  };
  auto fetch = [&](int c0) __attribute__((always_inline)) {
    if (s1 - c0 >= kCh) fetch_rows(c0, std::true_type{});
    else fetch_rows(c0, std::false_type{});
  };
  // Rows 16 j + 4 quad + i of the state are those of a 16 x 16 result, and a lane's of two of them make its eight k slots of a product:
  // rows of q and k lie in LDS in that order, four entries at a time. Result rows over tokens, 16 x + 4 quad + i, stand for token
  // 8 quad + 4 x + i: a lane's are eight in a row, and sums over tokens run in their order, from the most decayed on.
  auto place = [](int c) { return c < 4 ? 8 * c : 8 * (c - 4) + 4; };           // of the c-th four of 32
  const int kq_byte = 2 * (kq_d / 32 * 32 + place(kq_d % 32 / 4)), p_byte = p_tok * PB + 8 * (threadIdx.x & 7);
  const int r_tok = 8 * (r >> 2) + (r & 3), a_off = r_tok * RB + 16 * quad, m_off = r_tok * PB + 16 * quad;       // a lane's 16 bytes of a left-hand row
  // K^T comes transposed out of LDS: a lane names four entries of one token and gets one entry of four tokens
  const int t_off = (8 * quad + (r >> 2)) * RB + 16 * (r & 3);
  auto frag = [&](const unsigned char* at) __attribute__((always_inline)) {
    return __builtin_bit_cast(chunk_bf16x8, *reinterpret_cast<const uint4*>(at));
  };
  auto frag_t = [&](const unsigned char* img, int j) __attribute__((always_inline)) {
    using lds_bf16x4 = __attribute__((address_space(3))) chunk_bf16x4;
    const unsigned char* at = img + t_off + 64 * (j >> 1) + 8 * (j & 1);
    const chunk_bf16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)at);
    const chunk_bf16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(at + 4 * RB));
    return chunk_bf16x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
  };
  auto mm = [](chunk_bf16x8 a, chunk_bf16x8 bb, f32x4 c) __attribute__((always_inline)) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bb, c, 0, 0, 0);
  };
  auto rows4 = [&](const float* from, int x) __attribute__((always_inline)) {   // of a vector over tokens
    return *reinterpret_cast<const float4*>(from + 8 * quad + 4 * x);
  };
  auto scale4 = [&](f32x4 x, float4 f) __attribute__((always_inline)) { return f32x4{x[0] * f.x, x[1] * f.y, x[2] * f.z, x[3] * f.w}; };
  const f32x4 zero{0.0f, 0.0f, 0.0f, 0.0f};
  auto cut8 = [](f32x4 a, f32x4 c, chunk_bf16x8 (&to)[3]) __attribute__((always_inline)) {
    const Pieces4 x = cut4(a[0], a[1], a[2], a[3]), y = cut4(c[0], c[1], c[2], c[3]);
#pragma unroll
    for (int i = 0; i < 3; ++i) to[i] = join8(x.p[i], y.p[i]);
  };
  auto all_finite = [](const f32x4 (&x)[2]) __attribute__((always_inline)) {
    float z = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) z = fmaf(x[i >> 2][i & 3], 0.0f, z);
    return __builtin_amdgcn_ballot_w64(z != 0.0f) == 0;
  };
  // four entries from the place `at` on, put together from their pieces (an infinity's others are no numbers)
  auto matrix4 = [&](const unsigned char* at) {
    float4 x = ld4(reinterpret_cast<const bf16_t*>(at));
#pragma unroll
    for (int i = 1; i < 3; ++i) {
      const float4 y = ld4(reinterpret_cast<const bf16_t*>(at + i * kMatImg));
      auto add = [](float a, float c) { return __builtin_amdgcn_classf(a, 0x207) ? a : a + c; };
      x = float4{add(x.x, y.x), add(x.y, y.y), add(x.z, y.z), add(x.w, y.w)};
    }
    return x;
  };
  f32x4 U_next[2];
  auto stage = [&](int buf) __attribute__((always_inline)) {
    float z = 0.0f;                                    // NaN if a value is not finite
    auto put = [&](unsigned char* img, int at, uint2 v) __attribute__((always_inline)) {
      *reinterpret_cast<uint2*>(img + at) = v;
      auto hi = [](uint32_t x) { return __builtin_bit_cast(float, x & 0xffff0000u); };
      auto lo = [](uint32_t x) { return __builtin_bit_cast(float, x << 16); };
      z = fmaf(lo(v.x), 0.0f, fmaf(hi(v.x), 0.0f, fmaf(lo(v.y), 0.0f, fmaf(hi(v.y), 0.0f, z))));
    };
#pragma unroll
    for (int it = 0; it < KQ; ++it) {
      const int at = (kq_tok + it * (NT / (D / 4))) * RB + kq_byte;
      put(k_all[buf], at, kreg[it]);
      if constexpr (FULL) put(q_all[buf], at, qreg[it]);
    }
#pragma unroll
    for (int it = 0; it < PN; ++it) {
      const int m = (it * NT + (w << 6)) >> 8;
      if (m < MATS) {
        const float4 x = preg[it];
        z = fmaf(x.x, 0.0f, fmaf(x.y, 0.0f, fmaf(x.z, 0.0f, fmaf(x.w, 0.0f, z))));
        const Pieces4 c = cut4(x.x, x.y, x.z, x.w);
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<uint2*>(p_all[buf][m] + i * kMatImg + p_byte) = c.p[i];
      }
    }
    const bool odd = __builtin_amdgcn_ballot_w64(z != 0.0f) != 0;
    if (lane == 0) odd_all[buf][w] = odd;
#pragma unroll
    for (int i = 0; i < 8; ++i) U_next[i >> 2][i & 3] = __builtin_bit_cast(float, vreg[i] << 16);
    if (w % WPW == 0) ge_all[buf][hw][lane] = gereg;
  };
  // Two buffers: a chunk is staged while the one before it is computed, each wave at its own time, and two chunks ahead are on
  // their way in registers. One barrier a chunk.
  fetch(s0);
  stage(0);
  if (s0 + kCh < s1) fetch(s0 + kCh);
  __syncthreads();
  int buf = 0;
  for (int c0 = s0; c0 < s1; c0 += kCh, buf ^= 1) {
    const int cn = min(kCh, s1 - c0);
    const unsigned char *k_lds = k_all[buf], *q_lds = q_all[buf], *p_lds = p_all[buf][MATS > 0 ? hw : 0];
    const float* ge_lds = ge_all[buf][hw];
    const f32x4 U[2] = {U_next[0], U_next[1]};
    if constexpr (!FULL) {                             // (few products to stand among: 85 us there, 68 here, in the launch of 323)
      stage(buf ^ 1);
      if (c0 + 2 * kCh < s1) fetch(c0 + 2 * kCh);
    }
    f32x4 o[2], u2[2], next[DT];
#pragma unroll
    for (int x = 0; x < 2; ++x) u2[x] = scale4(U[x], rows4(ge_lds + kCh, x));
    const float g_last = ge_lds[cn - 1];
    bool odd = __builtin_amdgcn_ballot_w64(odd_all[buf][lane & (NW - 1)] != 0) != 0 || !all_finite(u2) || (FULL && !all_finite(U));
    if (__builtin_expect(!odd, 1)) {
      f32x4 qs[2][2], pu[2];                           // [sum][rows]: the largest pieces' products apart from the others'
#pragma unroll
      for (int x = 0; x < 2; ++x) qs[0][x] = qs[1][x] = pu[x] = zero;
      chunk_bf16x8 uc[3];
      cut8(u2[0], u2[1], uc);
      if constexpr (FULL) stage(buf ^ 1);
#pragma unroll
      for (int jj = 0; jj < DT / 2; ++jj) {
        if constexpr (FULL) {
          chunk_bf16x8 sc[3];
          cut8(S[2 * jj], S[2 * jj + 1], sc);
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const chunk_bf16x8 qf = frag(q_lds + 4 * x * RB + 64 * jj + a_off);
            qs[1][x] = mm(qf, sc[2], qs[1][x]);
            qs[1][x] = mm(qf, sc[1], qs[1][x]);
            qs[0][x] = mm(qf, sc[0], qs[0][x]);
          }
        }
#pragma unroll
        for (int j = 2 * jj; j < 2 * jj + 2; ++j) {
          const chunk_bf16x8 kf = frag_t(k_lds, j);
          f32x4 rest = mm(kf, uc[1], mm(kf, uc[2], zero));
#pragma unroll
          for (int i = 0; i < 4; ++i) rest[i] = fmaf(S[j][i], g_last, rest[i]);
          next[j] = mm(kf, uc[0], rest);
        }
      }
      if constexpr (FULL) {
        // U as it came: bf16
        const chunk_bf16x8 ub = join8(uint2{high_halves(U[0][0], U[0][1]), high_halves(U[0][2], U[0][3])},
                                      uint2{high_halves(U[1][0], U[1][1]), high_halves(U[1][2], U[1][3])});
#pragma unroll
        for (int x = 0; x < 2; ++x) {
#pragma unroll
          for (int i = 2; i >= 0; --i) pu[x] = mm(frag(p_lds + i * kMatImg + 4 * x * PB + m_off), ub, pu[x]);
          o[x] = scale4(qs[0][x] + qs[1][x], rows4(ge_lds, x)) + skip * U[x] + pu[x];
        }
        odd = !all_finite(o);                          // the state itself may hold an infinity
      }
    } else if constexpr (FULL) {
      stage(buf ^ 1);
    }
    if (FULL && c0 + 2 * kCh < s1) fetch(c0 + 2 * kCh);
    if (__builtin_expect(odd, 0)) {
      // the chunk in f32, the lower triangle token by token: a value that is not finite would reach the tokens before it through zeros
      auto row4 = [&](const unsigned char* img, int tok, int d) {
        return ld4(reinterpret_cast<const bf16_t*>(img + tok * RB + 64 * (d / 32) + 2 * place(d % 32 / 4)));
      };
      if constexpr (FULL) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          f32x4 acc = zero;
#pragma unroll
          for (int j = 0; j < DT; ++j) {
            const float4 a = row4(q_lds, r_tok + 4 * x, 16 * j + 4 * quad);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, S[j][0], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, S[j][1], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, S[j][2], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, S[j][3], acc, 0, 0, 0);
          }
          o[x] = scale4(acc, rows4(ge_lds, x)) + skip * U[x];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll 1
          for (int from = 0; from < 4; ++from) {
            const int j = 8 * from + i;
            const float v = __shfl(U[i >> 2][i & 3], 16 * from + r, kWave);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
              const int t = 8 * quad + k;
              const float4 row = matrix4(p_lds + t * PB + 8 * (j / 4));
              const float e = (j & 2) ? ((j & 1) ? row.w : row.z) : ((j & 1) ? row.y : row.x);
              o[k >> 2][k & 3] = j <= t ? fmaf(e, v, o[k >> 2][k & 3]) : o[k >> 2][k & 3];
            }
          }
      }
#pragma unroll
      for (int j = 0; j < DT; ++j) {
        f32x4 add = S[j] * g_last;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float4 row = row4(k_lds, 8 * quad + i, 16 * j + (r & 12));
          const float e = (r & 2) ? ((r & 1) ? row.w : row.z) : ((r & 1) ? row.y : row.x);
          add = __builtin_amdgcn_mfma_f32_16x16x4f32(e, u2[i >> 2][i & 3], add, 0, 0, 0);
        }
        next[j] = add;
      }
    }
#pragma unroll
    for (int j = 0; j < DT; ++j) S[j] = next[j];
    if constexpr (FULL) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i + 8 * quad < cn) p.o[(row0 + static_cast<int64_t>(c0 + i) * p.H + h) * p.Dv + o_off] = o[i >> 2][i & 3];
    }
    if constexpr (MODE == 1) seg_dec *= static_cast<double>(g_last);      // (only whole chunks)
    __syncthreads();                                   // the next chunk is complete, and nobody reads this one any more
  }
  if (MODE == 1 || s1 == n_all) {
    float* to = MODE == 1 ? gbase : sbase;
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) to[(16 * j + i) * p.Dv + st_off] = S[j][i];
  }
  if (MODE == 1 && lane == 0) p.seg_decay[(static_cast<int64_t>(b) * p.segs + blockIdx.y) * p.H + h] = static_cast<float>(seg_dec);
}

// seg_state: what each segment adds -> the state that each segment starts from. A thread owns four entries of a head's state.
__global__ __launch_bounds__(256) void chunk_combine_kernel(ChunkParams p) {
  const int b = blockIdx.z, h = blockIdx.y;
  const int n = p.cu_q[b + 1] - p.cu_q[b];
  const int segs = (n + p.seg_len - 1) / p.seg_len;
  const int64_t size = static_cast<int64_t>(p.D) * p.Dv;
  const int64_t x = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * 4;
  if (x >= size) return;
  float4 s{0, 0, 0, 0};
  if (p.ctx_lens[b] > 0) s = ld4(p.state + (static_cast<int64_t>(p.slots[b]) * p.H + h) * size + x);
  for (int i = 0; i < segs; ++i) {
    float* at = p.seg_state + ((static_cast<int64_t>(b) * p.segs + i) * p.H + h) * size + x;
    const bool last = i + 1 == segs;
    const float4 add = last ? float4{0, 0, 0, 0} : ld4(at);
    const float d = last ? 0.0f : p.seg_decay[(static_cast<int64_t>(b) * p.segs + i) * p.H + h];
    st4(at, s);
    s = float4{d * s.x + add.x, d * s.y + add.y, d * s.z + add.z, d * s.w + add.w};
  }
}

template <typename T, int KIND, int DT, int NW, int HPW, bool OWN = false>
static void chunk_launch(const ChunkParams& p, int B, hipStream_t s) {
  dim3 grid(p.H / HPW * (p.Dv / 16 / (NW / HPW)), p.segs, B), block(NW * 64);
  auto scan = [&](auto mode) {
    if constexpr (KIND == kChunkStep) chunk_step_kernel<DT, NW, HPW, decltype(mode)::value><<<grid, block, 0, s>>>(p);
    else chunk_scan_kernel<T, KIND, DT, NW, HPW, decltype(mode)::value, false, OWN><<<grid, block, 0, s>>>(p);
  };
  if (p.segs <= 1) {
    scan(std::integral_constant<int, 0>{});
    return;
  }
  if constexpr (KIND != kChunkDelta) {
    scan(std::integral_constant<int, 1>{});
    chunk_combine_kernel<<<dim3((p.D * p.Dv / 4 + 255) / 256, p.H, B), dim3(256), 0, s>>>(p);
    scan(std::integral_constant<int, 2>{});
  }
}

// Sequences, or segments of them at most.
static int64_t chunk_pieces(int64_t tokens, int B, int segs, int seg_len) {
  return segs > 1 ? std::min<int64_t>(static_cast<int64_t>(B) * segs, tokens / seg_len + B) : B;
}

static bool chunk_few(int64_t pieces, int H, int Dv) { return pieces * H * Dv / 128 <= 128; }

// Whether a launch of constant decays forms P in the scan (OWN), without a launch in front of it: q k^T of a chunk is 5 % more of the chain, and
// the powers of the decay are the same in every chunk. 16 x 1024 tokens, 16 heads of 128, the layer 803 -> 774 us (61 us in front, the silu of q and
// k once more and 67 MB through memory; 781 with q k^T in front of the staging). Scans by themselves, us, launch in front / OWN:
//   few workgroups wait for the longer chain: one prompt of 1000 138 / 144.
//   128 x 128, 16 heads: 16 x 1024 292 / 268, 64 x 250 304 / 287, 256 x 64 393 / 379; 16 of 290 to 1680 421 / 421; not where one sequence is what the
//     others are waiting for (one of 4000 beside 12 of 300 871 / 949).
//   128 x 64: three chunks of q and k in LDS leave a compute unit one workgroup of four waves instead of two: 256 x 64 231 / 301, 11 x 1500, 32 heads,
//     503 / 555; one of 4096 in segments 164 / 169.
//   keys of 64: two workgroups of four waves instead of three, and a chain of its own in front of the first chunk. Even lengths gain,
//     64 x 64, 32 heads, 16 x 1024 249 / 208, 128 x 120 243 / 236; 64 x 128, 16 heads, 188 / 179, 213 / 214; so do launches of one round that is
//     not mostly idle behind its longest (64 heads of 64 x 64, 8 of 20 to 220 45 / 39). In several rounds two chunks a sequence
//     lose (256 x 64 259 / 266 and 246 / 256), and so do uneven lengths (24 of 30 to 509 145 / 152; one of 4000 beside 12 of 300 453 / 522).
// Random steps that the rule takes, of 329 for each size: 1.04 times faster in the mean (128 x 128; the slowest 0.98), 1.07 (64 x 64; 0.98) and 1.03 (64 x 128; 0.98).
static bool chunk_own(int kind, int64_t tokens, int B, int max_new, int H, int D, int Dv, int segs, int seg_len) {
  const int64_t pieces = chunk_pieces(tokens, B, segs, seg_len), longest = segs > 1 ? seg_len : max_new, columns = static_cast<int64_t>(H) * Dv;
  if (kind != kChunkConst || chunk_few(pieces, H, Dv)) return false;
  if (D == 128) return Dv % 128 == 0 && longest * pieces <= 3 * tokens;
  const bool one_round = pieces * columns <= 256 * 128 && 5 * tokens * columns >= 2 * 256 * 128 * longest;      // 256 workgroups of 128 columns, 0.4 of them at work
  return one_round || (tokens >= 96 * pieces && 2 * longest * pieces <= 3 * tokens);
}

// Eight waves a workgroup: 128 columns of a head, or two heads of 64 that share q and k. Launches of few workgroups, which leave half of the
// chip empty, cut them in two (the f32 scans: a compute unit then holds one wave a SIMD, and a chunk takes two thirds of the time, though q
// and k are staged twice); beyond that the halves only take each other's place. us, 8 / 4 waves, 16 heads of 128 x 128, prompts of 1000: delta
// rule 1 prompt 268 / 186, 8 284 / 207, 10 294 / 384; constant decays 228 / 168, 253 / 194, 259 / 294; heads of 64 x 64, delta rule, 12
// prompts 204 / 150. Step sizes are bound by a chunk's chain either way (one prompt of 4096, 32 heads of 128 x 64, 469 / 500).
template <typename T, int KIND, int DT>
static void chunk_waves(const ChunkParams& p, int64_t tokens, int B, bool own, hipStream_t s) {
  constexpr bool CONST = KIND == kChunkConst;
  if constexpr (CONST) {
    if (own) {
      if constexpr (DT == 4) {
        if (p.Dv == 64) return chunk_launch<T, KIND, DT, 4, 1, true>(p, B, s);
      }
      return chunk_launch<T, KIND, DT, 8, 1, true>(p, B, s);
    }
  }
  chunk_prep_kernel<T, KIND, DT * 16><<<dim3(static_cast<unsigned>(tokens / kCh + B), p.G), dim3(256), 0, s>>>(p);
  const bool few = KIND != kChunkStep && chunk_few(chunk_pieces(tokens, B, p.segs, p.seg_len), p.H, p.Dv);
  if (p.Dv % 128 == 0 && !few) return chunk_launch<T, KIND, DT, 8, 1>(p, B, s);
  if constexpr (!CONST) {                              // (heads of the layers share no q and k; others take four waves)
    if (p.Dv % 128 != 0 && p.H / p.G % 2 == 0 && !few) return chunk_launch<T, KIND, DT, 8, 2>(p, B, s);
  }
  chunk_launch<T, KIND, DT, 4, 1>(p, B, s);
}

// The delta rule with norm and gate: heads of 64 or 128 values, on eight waves.
template <int DT>
static void chunk_norm_launch(const ChunkParams& p, int B, hipStream_t s) {
  if (p.Dv == 128) chunk_scan_kernel<float, kChunkDelta, DT, 8, 1, 0, true><<<dim3(p.H, 1, B), dim3(512), 0, s>>>(p);
  else chunk_scan_kernel<float, kChunkDelta, DT, 8, 2, 0, true><<<dim3(p.H / 2, 1, B), dim3(512), 0, s>>>(p);
}

static void chunk_norm_dispatch(const ChunkParams& p, int64_t tokens, int B, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(tokens / kCh + B), p.G), block(256);
  if (p.D == 64) {
    chunk_prep_kernel<float, kChunkDelta, 64><<<grid, block, 0, s>>>(p);
    chunk_norm_launch<4>(p, B, s);
  } else {
    chunk_prep_kernel<float, kChunkDelta, 128><<<grid, block, 0, s>>>(p);
    chunk_norm_launch<8>(p, B, s);
  }
}

template <typename T, int KIND>
static void chunk_dispatch(const ChunkParams& p, int64_t tokens, int B, bool own, hipStream_t s) {
  if (p.D == 64) chunk_waves<T, KIND, 4>(p, tokens, B, own, s);
  else chunk_waves<T, KIND, 8>(p, tokens, B, own, s);
}

static int chunk_segments(int kind, int max_new, int seg_len) {
  return kind == kChunkDelta || seg_len <= 0 || max_new <= seg_len ? 1 : (max_new + seg_len - 1) / seg_len;
}

static bool chunk_sizes_ok(int H, int G, int D, int Dv) {
  return H > 0 && G > 0 && H % G == 0 && (D == 64 || D == 128) && (Dv == 64 || (Dv > 0 && Dv % 128 == 0));
}

}  // namespace lvmix

using namespace lvmix;

extern "C" {

int64_t lv_chunk_scan_workspace_bytes(int kind, int64_t T, int B, int max_new, int H, int D, int Dv, int seg_len) {
  if (T < 0 || B < 0 || H <= 0 || D <= 0 || Dv <= 0 || max_new < 0) return fail(-1, "lv_chunk_scan_workspace_bytes: bad sizes");
  const int64_t rows = T * H;
  const int segs = chunk_segments(kind, max_new, seg_len);
  int64_t floats = chunk_own(kind, T, B, max_new, H, D, Dv, segs, seg_len) ? 0 : rows * kCh * (kind == kChunkDelta ? 2 : 1) + 2 * ((rows + 3) / 4 * 4);
  if (segs > 1) floats += static_cast<int64_t>(B) * segs * H * (static_cast<int64_t>(D) * Dv + 1);
  return floats * static_cast<int64_t>(sizeof(float));
}

static int chunk_scan(int kind, const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv, const void* a,
                      int64_t lda, const void* decay, const void* p0, const void* p1, const void* p2, void* state,
                      const int32_t* cu_q, const int32_t* ctx_lens, const int32_t* slots, void* o, void* workspace,
                      int64_t workspace_bytes, int64_t T, int B, int max_new, int H, int G, int D, int Dv, int seg_len,
                      const ChunkParams* norm, void* stream) {
  if (B == 0 || T == 0) return 0;
  if (!q || !k || !v || !state || !cu_q || !ctx_lens || !slots || !o) return fail(-1, "lv_chunk_scan: null pointer");
  if (kind != kChunkStep && kind != kChunkConst && kind != kChunkDelta) return fail(-1, "lv_chunk_scan: kind %d", kind);
  if (kind == kChunkStep && (!a || !p0 || !p1 || !p2)) return fail(-1, "lv_chunk_scan: step sizes without their parameters");
  if (kind != kChunkStep && (!decay || (kind == kChunkDelta && !a))) return fail(-1, "lv_chunk_scan: no decays");
  if (B < 0 || T < 0 || max_new <= 0 || max_new > T || seg_len < 0 || seg_len % kCh != 0 || !chunk_sizes_ok(H, G, D, Dv))
    return fail(-1, "lv_chunk_scan: bad sizes");
  const uintptr_t piece = kind == kChunkDelta ? 16 : 8;      // four entries of a row: f32 for the delta rule, bf16 otherwise
  if (ldq < static_cast<int64_t>(G) * D || ldk < static_cast<int64_t>(G) * D || ldv < static_cast<int64_t>(H) * Dv ||
      (kind == kChunkStep && lda < H) || ldq % 4 != 0 || ldk % 4 != 0 ||
      reinterpret_cast<uintptr_t>(q) % piece != 0 || reinterpret_cast<uintptr_t>(k) % piece != 0 ||
      reinterpret_cast<uintptr_t>(state) % 16 != 0 || reinterpret_cast<uintptr_t>(workspace) % 16 != 0)
    return fail(-1, "lv_chunk_scan: strides or alignment");
  const int64_t need = lv_chunk_scan_workspace_bytes(kind, T, B, max_new, H, D, Dv, seg_len);
  if (need > 0 && !workspace) return fail(-1, "lv_chunk_scan: null pointer");
  if (workspace_bytes < need)
    return fail(-3, "lv_chunk_scan: workspace of %lld bytes", static_cast<long long>(workspace_bytes));
  const int64_t rows = T * H, rows4 = (rows + 3) / 4 * 4;
  float* ws = static_cast<float*>(workspace);
  ChunkParams p{q, k, v, ldq, ldk, ldv, a, lda, static_cast<const float*>(decay), static_cast<const float*>(p0),
                static_cast<const float*>(p1), static_cast<const float*>(p2), static_cast<float*>(state), cu_q, ctx_lens, slots,
                static_cast<float*>(o), nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, B, H, G, D, Dv, seg_len,
                chunk_segments(kind, max_new, seg_len)};
  const bool own = chunk_own(kind, T, B, max_new, H, D, Dv, p.segs, seg_len);
  if (!own) {
    p.P = ws;
    ws += rows * kCh;
    if (kind == kChunkDelta) {
      p.Tm = ws;
      ws += rows * kCh;
    }
    p.Gf = ws;
    p.Ef = ws + rows4;
    ws += 2 * rows4;
  }
  if (p.segs > 1) {
    p.seg_state = ws;
    p.seg_decay = ws + static_cast<int64_t>(B) * p.segs * H * D * Dv;
  }
  hipStream_t s = as_stream(stream);
  if (norm != nullptr) {
    p.gate = norm->gate;
    p.ld_gate = norm->ld_gate;
    p.norm_w = norm->norm_w;
    p.eps = norm->eps;
    p.gate_silu = norm->gate_silu;
    chunk_norm_dispatch(p, T, B, s);
  } else if (kind == kChunkDelta) chunk_dispatch<float, kChunkDelta>(p, T, B, false, s);
  else if (kind == kChunkStep) chunk_dispatch<bf16_t, kChunkStep>(p, T, B, false, s);
  else chunk_dispatch<bf16_t, kChunkConst>(p, T, B, own, s);
  return launched("lv_chunk_scan");
}

int lv_chunk_scan(int kind, const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv, const void* a,
                  int64_t lda, const void* decay, const void* p0, const void* p1, const void* p2, void* state,
                  const int32_t* cu_q, const int32_t* ctx_lens, const int32_t* slots, void* o, void* workspace,
                  int64_t workspace_bytes, int64_t T, int B, int max_new, int H, int G, int D, int Dv, int seg_len,
                  void* stream) {
  return chunk_scan(kind, q, ldq, k, ldk, v, ldv, a, lda, decay, p0, p1, p2, state, cu_q, ctx_lens, slots, o, workspace, workspace_bytes, T, B,
                    max_new, H, G, D, Dv, seg_len, nullptr, stream);
}

int lv_chunk_delta_norm(const void* q, const void* k, const void* v, const void* beta, const void* decay, void* state, const int32_t* cu_q,
                        const int32_t* ctx_lens, const int32_t* slots, const void* gate, int64_t ld_gate, const void* norm_w, void* out,
                        void* workspace, int64_t workspace_bytes, int64_t T, int B, int max_new, int H, int G, int D, int Dv, float eps,
                        int gate_kind, void* stream) {
  if (B == 0 || T == 0) return 0;
  if (!gate || !norm_w || (gate_kind != LV_MIX_GATE_SILU && gate_kind != LV_MIX_GATE_SIGMOID))
    return fail(-1, "lv_chunk_delta_norm: gate, norm weight or gate kind %d", gate_kind);
  if ((Dv != 128 && (Dv != 64 || G <= 0 || H / G % 2 != 0)) || ld_gate < static_cast<int64_t>(H) * Dv || ld_gate >= (int64_t{1} << 27))
    return fail(-1, "lv_chunk_delta_norm: heads of %d values, gate rows of stride %lld", Dv, static_cast<long long>(ld_gate));
  ChunkParams norm{};
  norm.gate = static_cast<const bf16_t*>(gate);
  norm.ld_gate = ld_gate;
  norm.norm_w = static_cast<const float*>(norm_w);
  norm.eps = eps;
  norm.gate_silu = gate_kind == LV_MIX_GATE_SILU;
  const int64_t gd = static_cast<int64_t>(G) * D;
  return chunk_scan(kChunkDelta, q, gd, k, gd, v, static_cast<int64_t>(H) * Dv, beta, 0, decay, nullptr, nullptr, nullptr, state, cu_q, ctx_lens,
                    slots, out, workspace, workspace_bytes, T, B, max_new, H, G, D, Dv, 0, &norm, stream);
}

}  // extern "C"
