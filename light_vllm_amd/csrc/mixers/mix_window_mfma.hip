// Matrix-core form of the windowed pooled attention for bf16 activations and caches.
//
// Steps of one token a sequence: decode_pool_kernel; prompts: prompt_attn_kernel; both below, for the usual head sizes. Here, for all others:
// One workgroup = one tile of 16 consecutive new tokens of one sequence, one kv head, up to four of its
// query heads (one per wave). Keys are walked in tiles of 64 entries, first the pooled blocks that any
// query of the tile may see, then the tokens from the first window start to the last query; what a
// query does not see (outside its window, a block not yet wholly before it, the future) is masked.
//
// Everything is computed transposed so that no operand changes layout between the two products:
//   S^T = K Q^T   v_mfma_f32_16x16x32_bf16, A = 16 keys x 32 of D read straight from the cache rows with 16-byte loads, B = the
//                 wave's Q fragments (registers, loaded once); a lane ends up with 4 keys of ONE query, so the softmax
//                 statistics of a query live in 4 lanes (two shuffles) and
//   O^T += V^T P^T  takes the probabilities of two 16-key blocks as its B operand exactly as they lie (keys x
//                 queries), with A = V^T from transposing LDS reads of the 64-entry V tile that the four waves stage
//                 together, rows as they are.
// Fragment counts are compile-time bounds and nothing in the tile loop branches on the head sizes: a step past the end of D reads
// the last entries of the row again against zeros in Q, a block past Dv reads the last block of V and is not stored. (With a
// branch around every load and its MFMA the loads could not be issued together, and the kernel ran at one memory latency per
// MFMA.)
// The sink is the initial state of the running softmax: maximum 0 (or the head's learned number), sum 1.
// Extended form: a tile's key factors (norms kept beside unnormed keys) and the heads' distance biases sit in LDS; a score becomes
// product * scale * factor + bias before the softmax.
#include "mix_common.h"

#include <algorithm>

namespace lvmix {

typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4v_t;
typedef __attribute__((address_space(3))) __bf16 lds_bf16;
typedef __attribute__((address_space(3))) bf16x4v_t lds_bf16x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

struct WindowMfmaParams {
  const uint16_t *q, *k_cache, *v_cache, *kp, *vp, *gate;
  int64_t ld_gate;
  int gate_dv;         // entries of a gate row per head: Dv (one per output channel) or 1 (one per head)
  uint16_t* out;
  const int32_t *cu_q, *ctx_lens, *block_tables;
  int bt_stride, H, G, D, Dv, page, window, P, PP, ngroups;
  float scale, sink;
  uint32_t m_page, m_P, m_nseg;   // floor(2^32 / d) of the three divisors the tile loop divides by (see fdiv)
  int nsplit;          // > 1 (launches of at most one query tile per sequence): grid.x = split of the key tiles
  float* ws;           // [T, H, nsplit, Dv + 4] partial read-outs, running maximum and sum
  int64_t k_ld, v_ld;  // elements between the rows of two cached tokens (G*D, G*Dv unless the caches are views of wider rows)
  float m0;            // start of the running maximum: the sink's score 0, or far below any score without a sink
  int keep_first;      // positions below this are seen from everywhere; they take the place of the pooled tiles (P == 0)
  int chunk;           // > 0: a query sees its own chunk of that many positions (counted from 0) up to itself; no window
  const float* sinks;  // [H] or NULL: a learned score per query head in place of the sink's 0
  float cap_in, cap;   // kCapped: scores pass cap * tanh(product * cap_in), cap_in = scale / cap
  const float* key_scale;   // kExtended: [pages, page, G] or NULL, a factor on the score of every cached key
  const float* dist_bias;   // kExtended: [H, bias_len] or NULL, added to the score at distance min(pos - key, bias_len - 1)
  int bias_len;
  int64_t out_ld;      // elements between the output rows of two tokens
};

enum ScoreForm { kPlain = 0, kCapped = 1, kExtended = 2 };

// Latent attention with its two matrices in the attention kernel: q holds the heads' own queries, [T, H, Dn + Dr], and out their own
// outputs, [T, H, Dn]; D = R + Dr and Dv = R stay those of the cached rows.
struct LatentParams : WindowMfmaParams {
  const uint16_t *uk, *uv;   // [H, Dn, R], [H, R, Dn]
  const float* inv_freq;     // [Dr / 2]
};

constexpr int kTileQ = 16;
constexpr int kTileK = 64;
constexpr int kMaxK32 = 8;     // D <= 256: 32-wide steps over D (template K32: 2, 4 or 8)
// Row stride of the V tile: an odd multiple of 16 entries, so that the 16 rows a transposed read touches lie in all banks.
__host__ __device__ constexpr int v_row(int Dv) { return Dv % 32 == 0 ? Dv + 16 : Dv; }
constexpr int kMaxDvb = 16;    // Dv <= 256
constexpr int kBiasLds = 1024; // distance biases of a head up to this many are copied to LDS (longer tables are read from memory)
constexpr int kBtCache = 2048; // page ids of a sequence kept in LDS (longer sequences look them up in memory)

// n / d for 0 <= n < 2^31 with magic = floor(2^32 / d) (0xffffffff for d = 1): the estimate is the quotient or one
// less. The tile loop divides by the page size, the pool size and the row's segment count for every row address;
// the compiler's general 32-bit division is some forty instructions each and dominated the kernel.
__device__ __forceinline__ int fdiv(int n, int d, uint32_t magic) {
  const uint32_t q = __umulhi(static_cast<uint32_t>(n), magic);
  const uint32_t r = static_cast<uint32_t>(n) - q * static_cast<uint32_t>(d);
  return static_cast<int>(r >= static_cast<uint32_t>(d) ? q + 1 : q);
}

__device__ __forceinline__ short bf16_bits(float x) {
  __bf16 b = static_cast<__bf16>(x);
  return __builtin_bit_cast(short, b);
}

// tanh through the exponential: the absolute error stays at a few 1e-7, which is what a score multiplied by the cap needs.
__device__ __forceinline__ float fast_tanh(float x) { return 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + __expf(2.0f * x)); }

// AHEAD: the next tile's V rows, key-row addresses and (once the current scores are done) K fragments are fetched while
// the current tile is computed. That pays when a launch has few workgroups per compute unit (decoded tokens). A prompt's
// many tiles hide latency by occupancy instead, and every register counts there: with the 32 registers of a V tile held
// ahead the kernel fell from two waves a SIMD to one and ran 1.7x slower; K32 and DVB size the fragment arrays for the
// head sizes at hand for the same reason.
template <bool AHEAD, int K32, int DVB, int FORM>
__global__ __launch_bounds__(256, AHEAD ? 1 : (DVB > 8 ? 2 : (DVB > 4 ? 3 : 4))) void window_pool_mfma_kernel(WindowMfmaParams p) {
  extern __shared__ __attribute__((aligned(16))) uint16_t vs[];             // V tile [kTileK][ldv]
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int ln = lane & 15, lg = lane >> 4;
  const int b = blockIdx.z;
  const int g = blockIdx.y / p.ngroups, hg = blockIdx.y % p.ngroups;
  const int q0 = p.cu_q[b], n = p.cu_q[b + 1] - q0;
  const int split = p.nsplit > 1 ? blockIdx.x : 0;
  const int r0 = p.nsplit > 1 ? 0 : blockIdx.x * kTileQ;
  if (r0 >= n) return;
  const int ctx = p.ctx_lens[b];
  const int nvalid = min(kTileQ, n - r0);
  const int i0 = ctx + r0, i1 = i0 + nvalid - 1;
  const bool qvalid = ln < nvalid;
  const int r = r0 + min(ln, nvalid - 1);
  const int pos = ctx + r;
  const int64_t t = q0 + r;
  const int rep = p.H / p.G;
  const int hloc = hg * 4 + wave;
  const bool active = hloc < rep;
  const int h = g * rep + min(hloc, rep - 1);
  const int D = p.D, Dv = p.Dv, page = p.page, P = p.P, W = p.window;
  const int ndvb = Dv / 16, ldv = v_row(Dv);
  // transposed reads: of every 4 keys x 16 columns, lane 4 q + r of 16 names key q, columns 4r .. 4r + 3, and gets column 4 q + r of all four
  const lds_bf16* vt0 = (const lds_bf16*)vs + (4 * lg + (ln >> 2)) * ldv + 4 * (ln & 3);
  const int64_t GD = static_cast<int64_t>(p.G) * D, GDv = static_cast<int64_t>(p.G) * Dv;
  const int32_t* bt_global = p.block_tables + static_cast<int64_t>(b) * p.bt_stride;
  // the sequence's page ids up to the last query's page, once, so that no row address waits for a second trip to memory
  __shared__ int32_t bt_lds[kBtCache];
  const int nbt = (ctx + r0 + nvalid - 1) / page + 1;
  const bool bt_cached = nbt <= kBtCache;
  if (bt_cached) {
    for (int x = threadIdx.x; x < nbt; x += blockDim.x) bt_lds[x] = bt_global[x];
    __syncthreads();
  }
  auto bt = [&](int idx) { return bt_cached ? bt_lds[idx] : bt_global[idx]; };
  // kExtended: the tile's key factors and the distance biases of the workgroup's heads, behind the V tile
  float* ks_lds = reinterpret_cast<float*>(vs + kTileK * ldv);             // [kTileK]
  float* bias_lds = ks_lds + kTileK;                                       // [4][bias_len]
  const float* bias_h = nullptr;
  float bias_reg[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  bool bias_cached = false;
  if constexpr (FORM == kExtended) {
    if (p.dist_bias != nullptr) {
      bias_cached = p.bias_len <= kBiasLds;
      bias_h = p.dist_bias + static_cast<int64_t>(h) * p.bias_len;
#pragma unroll
      for (int x = 0; x < 4; ++x) bias_reg[x] = bias_h[min(lane + x * kWave, p.bias_len - 1)];     // stored behind the first tile's requests
    }
    if (p.key_scale == nullptr && threadIdx.x < kTileK) ks_lds[threadIdx.x] = 1.0f;                 // read behind the first barrier
  }

  bf16x8_t qf[K32];
  int koff[K32];                                        // this lane's entries of a key or query row in step kk
  {
    const uint16_t* qrow = p.q + (t * p.H + h) * D;
#pragma unroll
    for (int kk = 0; kk < K32; ++kk) {
      koff[kk] = min(32 * kk + 8 * lg, D - 8);
      qf[kk] = *reinterpret_cast<const bf16x8_t*>(qrow + koff[kk]);
      if (32 * kk + 8 * lg >= D) qf[kk] = __builtin_bit_cast(bf16x8_t, u32x4_t{0, 0, 0, 0});
    }
  }
  f32x4_t acc_o[DVB];
#pragma unroll
  for (int d = 0; d < DVB; ++d) acc_o[d] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  float m = p.sinks != nullptr ? p.sinks[h] : p.m0, l = split == 0 ? p.sink : 0.0f;

  const int chunk = p.chunk, keep = p.keep_first;
  const int jlo = chunk > 0 ? (i0 / chunk) * chunk : max(0, i0 - W + 1);
  const int cstart = chunk > 0 ? (pos / chunk) * chunk : 0;                // first position of this lane's query's chunk
  // entries of the first phase: pooled blocks the last query sees, or (without a pool) kept first tokens before the token tiles
  const int nbmax = P > 0 ? ((chunk == 0 && i1 - W + 1 > 0) ? (i1 - W + 1) / P : 0) : min(keep, jlo);

  // The tiles of both phases as one list: [pooled tiles | token tiles]. The V rows of the next tile and the
  // addresses of its key rows are fetched while the current tile is computed; they meet LDS behind a barrier.
  const int npt = (nbmax + kTileK - 1) / kTileK;
  const int ntt = (i1 + 1 - jlo + kTileK - 1) / kTileK;
  const int ntiles = npt + ntt;
  const int nseg = Dv / 8;                                                // 16-byte segments of a row

  auto tile_start = [&](int tile) { return tile < npt ? tile * kTileK : jlo + (tile - npt) * kTileK; };

  // Cache row of entry `lane` of a tile: every wave finds its 64 rows once, a lane each, and hands them round by shuffles.
  auto tile_slot = [&](int tile) {
    const int e = tile_start(tile) + lane;
    if (tile < npt && P > 0) {
      const int ec = min(e, nbmax - 1);
      const int pj = fdiv(ec * P + P - 1, page, p.m_page);
      return bt(pj) * p.PP + (ec - fdiv(page * pj, P, p.m_P));
    }
    const int ec = min(e, tile < npt ? nbmax - 1 : i1);
    const int pj = fdiv(ec, page, p.m_page);
    return bt(pj) * page + (ec - pj * page);
  };
  // V rows of a tile: consecutive threads take consecutive 16-byte segments of a row (whole cache lines per load instruction),
  // all of a thread's loads are issued together. AHEAD: one tile ahead of their use, and they wait in registers.
  constexpr int NV = DVB / 2;
  const bool keyed = FORM == kExtended && p.key_scale != nullptr && threadIdx.x < kTileK;
  float ksreg = 1.0f;
  u32x4_t vreg[NV];
  const uint16_t* knext[4];
  auto fetch_rows = [&](int tile) {
    const int slot = tile_slot(tile);
    const bool pooled = tile < npt && P > 0;
    const uint16_t* kbase = (pooled ? p.kp : p.k_cache) + g * D;
    const uint16_t* vbase = (pooled ? p.vp : p.v_cache) + g * Dv;
    const int64_t kld = pooled ? GD : p.k_ld, vld = pooled ? GDv : p.v_ld;
#pragma unroll
    for (int x = 0; x < NV; ++x) {
      const int c = min(static_cast<int>(threadIdx.x) + 256 * x, kTileK * nseg - 1);
      const int row = fdiv(c, nseg, p.m_nseg), seg = c - row * nseg;
      vreg[x] = *reinterpret_cast<const u32x4_t*>(vbase + __shfl(slot, row, kWave) * vld + seg * 8);
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) knext[kb] = kbase + __shfl(slot, kb * 16 + ln, kWave) * kld;
    if (keyed) ksreg = p.key_scale[static_cast<int64_t>(slot) * p.G + g];    // the first wave: lane = entry
  };
  // Only LDS traffic meets at the barriers of the tile loop. The fetch-ahead variant waits for that alone, so that the
  // vector loads of the next tile stay in flight across them (a full __syncthreads would drain them every tile).
  auto tile_barrier = [&]() {
    if (AHEAD) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else __syncthreads();
  };
  bf16x8_t kdata[AHEAD ? 4 : 1][K32];
  auto fetch_k = [&]() {                                                    // the K fragments of the tile knext points to
#pragma unroll
    for (int kb = 0; kb < (AHEAD ? 4 : 0); ++kb) {
#pragma unroll
      for (int kk = 0; kk < K32; ++kk) kdata[kb][kk] = *reinterpret_cast<const bf16x8_t*>(knext[kb] + koff[kk]);
    }
  };
  // a split takes a contiguous share of the tiles
  const int per_split = p.nsplit > 1 ? (ntiles + p.nsplit - 1) / p.nsplit : ntiles;
  const int t_begin = split * per_split, t_end = min(ntiles, t_begin + per_split);
  if (AHEAD && t_begin < t_end) {
    fetch_rows(t_begin);
    if (active) fetch_k();
  }
  if (bias_cached) {                                                       // read by this wave alone
#pragma unroll
    for (int x = 0; x < 4; ++x)
      if (lane + x * kWave < p.bias_len) bias_lds[wave * p.bias_len + lane + x * kWave] = bias_reg[x];
    for (int x = lane + 4 * kWave; x < p.bias_len; x += kWave) bias_lds[wave * p.bias_len + x] = bias_h[x];
  }
  for (int tile = t_begin; tile < t_end; ++tile) {
    const int phase = tile < npt ? 0 : 1;
    const int e0 = tile_start(tile);
    const int e_end = phase == 0 ? nbmax : i1 + 1;
    const uint16_t* kcur[4];
    tile_barrier();                                                         // the previous tile's V reads are done
    if constexpr (!AHEAD) fetch_rows(tile);
#pragma unroll
    for (int x = 0; x < NV; ++x) {
      const int c = threadIdx.x + 256 * x;
      if (c < kTileK * nseg) {
        const int row = fdiv(c, nseg, p.m_nseg), seg = c - row * nseg;
        *reinterpret_cast<u32x4_t*>(vs + row * ldv + seg * 8) = vreg[x];
      }
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) kcur[kb] = knext[kb];
    if (keyed) ks_lds[threadIdx.x] = ksreg;
    tile_barrier();
    if (AHEAD && tile + 1 < t_end) fetch_rows(tile + 1);
    if (!active) continue;
    {
      f32x4_t s[4];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const uint16_t* krow = kcur[kb];
        s[kb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kk = 0; kk < K32; ++kk)
          s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              AHEAD ? kdata[AHEAD ? kb : 0][kk] : *reinterpret_cast<const bf16x8_t*>(krow + koff[kk]), qf[kk], s[kb], 0, 0, 0);
      }
      if (AHEAD && tile + 1 < t_end) fetch_k();                            // in flight across the softmax, PV and the barriers
      // result row 4*lg + i of key block kb: key e0 + 16 kb + 4 lg + i
      if constexpr (FORM == kExtended) {
        const bool far = bias_h != nullptr && i0 - (e0 + kTileK - 1) >= p.bias_len - 1;      // all of the tile at the last bias
        const float bias_far = far ? (bias_cached ? bias_lds[wave * p.bias_len + p.bias_len - 1] : bias_h[p.bias_len - 1]) : 0.0f;
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          const f32x4_t ks = *reinterpret_cast<const f32x4_t*>(ks_lds + kb * 16 + 4 * lg);
          s[kb] = s[kb] * (ks * p.scale) + bias_far;
        }
        if (bias_h != nullptr && !far) {
#pragma unroll
          for (int kb = 0; kb < 4; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int dist = min(max(pos - (e0 + kb * 16 + 4 * lg + i), 0), p.bias_len - 1);
              s[kb][i] += bias_cached ? bias_lds[wave * p.bias_len + dist] : bias_h[dist];
            }
        }
      } else {
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) s[kb][i] = FORM == kCapped ? p.cap * fast_tanh(s[kb][i] * p.cap_in) : s[kb][i] * p.scale;
      }
      // a tile of tokens that every query of the workgroup sees whole needs no mask
      const bool whole = phase == 1 && e0 + kTileK - 1 <= i0 && (chunk > 0 ? e0 >= i1 - i1 % chunk : i1 - e0 < W);
      if (!whole) {
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int ke = e0 + kb * 16 + 4 * lg + i;
            bool vis = ke < e_end;
            if (phase == 0) vis = vis && (P == 0 || ke * P + P - 1 <= pos - W);
            else vis = vis && ke <= pos && ((chunk > 0 ? ke >= cstart : pos - ke < W) || ke < keep);
            s[kb][i] = vis ? s[kb][i] : -INFINITY;
          }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[kb][i]);
      mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
      mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
      const float nm = fmaxf(m, mx);
      const float corr = __expf(m - nm);
      float rs = 0.0f;
      bf16x8_t pb[2];                                                       // key blocks (0, 1) and (2, 3) side by side
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float e = __expf(s[kb][i] - nm);                            // exp(-inf) = 0 for what is not seen
          rs += e;
          pb[kb >> 1][(kb & 1) * 4 + i] = static_cast<__bf16>(e);
        }
      }
      rs += __shfl_xor(rs, 16, kWave);
      rs += __shfl_xor(rs, 32, kWave);
      l = l * corr + rs;
      m = nm;
#pragma unroll
      for (int d = 0; d < DVB; ++d) acc_o[d] *= corr;
#pragma unroll
      for (int c = 0; c < 2; ++c) {                                         // key blocks 2c and 2c + 1
#pragma unroll
        for (int d = 0; d < DVB; ++d) {
          const lds_bf16* vt = vt0 + 32 * c * ldv + 16 * min(d, ndvb - 1);
          const bf16x4v_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)vt);
          const bf16x4v_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vt + 16 * ldv));
          acc_o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), pb[c], acc_o[d], 0, 0, 0);
        }
      }
    }
  }
  if (!active || !qvalid) return;
  if (p.nsplit > 1) {                                                       // unnormalised partials; window_pool_merge_kernel ends the job
    float* w = p.ws + ((t * p.H + h) * p.nsplit + split) * (Dv + 4);
#pragma unroll
    for (int d = 0; d < DVB; ++d)
      if (d < ndvb)
        *reinterpret_cast<f32x4_t*>(w + 16 * d + 4 * lg) = acc_o[d];
    if (lg == 0) {
      w[Dv] = m;
      w[Dv + 1] = l;
    }
    return;
  }
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
  uint16_t* orow = p.out + t * p.out_ld + static_cast<int64_t>(h) * Dv;
  const uint16_t* grow = p.gate != nullptr ? p.gate + t * p.ld_gate + static_cast<int64_t>(h) * p.gate_dv : nullptr;
  const int gstep = p.gate_dv > 1 ? 1 : 0;
#pragma unroll
  for (int d = 0; d < DVB; ++d) {
    if (d < ndvb) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int dv = 16 * d + 4 * lg + i;
        float val = acc_o[d][i] * inv;
        if (grow != nullptr) val *= sigmoidf_(__builtin_bit_cast(float, static_cast<uint32_t>(grow[dv * gstep]) << 16));
        orow[dv] = static_cast<uint16_t>(bf16_bits(val));
      }
    }
  }
}

// One new token a sequence (decode steps), plain scores: up to 16 query heads of a kv head are the 16 columns of a product, so that a key
// row is read once for all of them; the kernel above gives every head a wave of its own, with one query in sixteen columns, and every wave the
// key rows. A wave walks tiles of 32 keys, the four waves of a workgroup and the splits share a sequence's tiles; waves meet in
// LDS, splits in window_pool_merge_kernel. Nothing but a tile's tail is masked: the one query sees every entry of the list. The rows of the next
// tile are requested as soon as the scores have used this one's registers. SAME: values are the first DV entries of the key rows and
// go from the registers to LDS, where they are read transposed.
// HBM-bound where there is enough to read, else a chain of loads: 48 sequences of 1100 tokens on average, 16 heads on latent rows of 192 + 64
// 123 -> 11 us (27 MB), 16 heads over 4 of 128 in a window of 1024 with pooled blocks 63 -> 24; 64 of 4000, 32 over 8, window 2048: 545 MB in
// 103 us; four of 1000 12.6 -> 5.9.
template <int DK, int DV, bool SAME>
__global__ __launch_bounds__(256, 2) void decode_pool_kernel(WindowMfmaParams p) {
  constexpr int KT = 32, NK = DK / 32, ND = DV / 16, LDV = v_row(DV), VN = SAME ? 1 : DV / 16;
  constexpr int IMAGE = KT * LDV * 2, PART = 16 * (DV + 4) * 4;
  constexpr int OWN = IMAGE > PART ? IMAGE : PART;
  __shared__ __attribute__((aligned(16))) unsigned char lds[4 * OWN];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, ln = lane & 15, lg = lane >> 4;
  const int b = blockIdx.z, g = blockIdx.y / p.ngroups, hg = blockIdx.y % p.ngroups, split = blockIdx.x;
  const int64_t t = p.cu_q[b];
  if (p.cu_q[b + 1] - static_cast<int>(t) <= 0) return;
  const int pos = p.ctx_lens[b], rep = p.H / p.G, P = p.P, page = p.page, chunk = p.chunk;
  const int h = g * rep + min(hg * 16 + ln, rep - 1);
  const int32_t* bt = p.block_tables + static_cast<int64_t>(b) * p.bt_stride;
  // the entries: pooled blocks or kept first tokens, then the window's or the chunk's tokens
  const int jlo = chunk > 0 ? pos / chunk * chunk : max(0, pos - p.window + 1);
  const int first = P > 0 ? (chunk == 0 && pos - p.window + 1 > 0 ? (pos - p.window + 1) / P : 0) : min(p.keep_first, jlo);
  const int npt = (first + KT - 1) / KT, ntiles = npt + (pos + 1 - jlo + KT - 1) / KT;
  const int per = (ntiles + p.nsplit - 1) / p.nsplit, end = min(ntiles, (split + 1) * per);

  bf16x8_t qf[NK];
#pragma unroll
  for (int kk = 0; kk < NK; ++kk) qf[kk] = *reinterpret_cast<const bf16x8_t*>(p.q + (t * p.H + h) * DK + 32 * kk + 8 * lg);
  f32x4_t o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) o[d] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  float m = fmaxf(p.sinks != nullptr ? p.sinks[h] : p.m0, -1e30f), l = split == 0 && wave == 0 ? p.sink : 0.0f;

  auto slot_of = [&](int tile) __attribute__((always_inline)) {             // cache row of entry `lane & 31`; past the end the last one's
    if (tile < npt) {
      const int e = min(tile * KT + (lane & 31), first - 1);
      if (P > 0) {
        const int pj = fdiv(e * P + P - 1, page, p.m_page);
        return bt[pj] * p.PP + (e - fdiv(page * pj, P, p.m_P));
      }
      const int pj = fdiv(e, page, p.m_page);
      return bt[pj] * page + (e - pj * page);
    }
    const int e = min(jlo + (tile - npt) * KT + (lane & 31), pos), pj = fdiv(e, page, p.m_page);
    return bt[pj] * page + (e - pj * page);
  };
  const int64_t GD = static_cast<int64_t>(p.G) * DK, GDv = static_cast<int64_t>(p.G) * DV;
  bf16x8_t kf[2][NK];
  u32x4_t vf[VN];
  auto request_k = [&](int tile, int slot) __attribute__((always_inline)) {
    const bool pooled = tile < npt && P > 0;
    const uint16_t* base = (pooled ? p.kp : p.k_cache) + g * DK + 8 * lg;
    const int64_t ld = pooled ? GD : p.k_ld;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const uint16_t* row = base + __shfl(slot, 16 * kb + ln, kWave) * ld;
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) kf[kb][kk] = *reinterpret_cast<const bf16x8_t*>(row + 32 * kk);
    }
  };
  auto request_v = [&](int tile, int slot) __attribute__((always_inline)) {
    if constexpr (!SAME) {
      const bool pooled = tile < npt && P > 0;
      const uint16_t* base = (pooled ? p.vp : p.v_cache) + g * DV + 8 * (lane % (DV / 8));
      const int64_t ld = pooled ? GDv : p.v_ld;
#pragma unroll
      for (int x = 0; x < VN; ++x)
        vf[x] = *reinterpret_cast<const u32x4_t*>(base + __shfl(slot, (512 / DV) * x + lane / (DV / 8), kWave) * ld);
    }
  };
  uint16_t* image = reinterpret_cast<uint16_t*>(lds + wave * OWN);
  const lds_bf16* vt = (const lds_bf16*)image + (4 * lg + (ln >> 2)) * LDV + 4 * (ln & 3);
  int tile = split * per + wave, slot = 0;
  if (tile < end) {
    slot = slot_of(tile);
    request_k(tile, slot);
    request_v(tile, slot);
    if (tile + 4 < end) slot = slot_of(tile + 4);
  }
  for (; tile < end; tile += 4) {
    f32x4_t s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      s[kb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kb][kk], qf[kk], s[kb], 0, 0, 0);
    }
    if constexpr (SAME) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int kk = 0; kk < DV / 32; ++kk)
          *reinterpret_cast<bf16x8_t*>(image + (16 * kb + ln) * LDV + 32 * kk + 8 * lg) = kf[kb][kk];
    } else {
#pragma unroll
      for (int x = 0; x < VN; ++x)
        *reinterpret_cast<u32x4_t*>(image + ((512 / DV) * x + lane / (DV / 8)) * LDV + 8 * (lane % (DV / 8))) = vf[x];
    }
    const int e0 = tile < npt ? tile * KT : jlo + (tile - npt) * KT, e_end = tile < npt ? first : pos + 1;
    if (tile + 4 < end) {
      request_k(tile + 4, slot);
      request_v(tile + 4, slot);
      if (tile + 8 < end) slot = slot_of(tile + 8);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[kb][i] = e0 + 16 * kb + 4 * lg + i < e_end ? s[kb][i] * p.scale : -INFINITY;
        mx = fmaxf(mx, s[kb][i]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    const float nm = fmaxf(m, mx), corr = __expf(m - nm);
    float rs = 0.0f;
    bf16x8_t pb;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = __expf(s[kb][i] - nm);                              // exp(-inf) = 0 for what is not there
        rs += e;
        pb[4 * kb + i] = static_cast<__bf16>(e);
      }
    rs += __shfl_xor(rs, 16, kWave);
    rs += __shfl_xor(rs, 32, kWave);
    l = l * corr + rs;
    m = nm;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      const bf16x4v_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vt + 16 * d));
      const bf16x4v_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vt + 16 * d + 16 * LDV));
      o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), pb, o[d] * corr, 0, 0, 0);
    }
  }
  // the waves' sums, [16 heads][DV | maximum, sum], each over its own image
  float* part = reinterpret_cast<float*>(lds + wave * OWN) + ln * (DV + 4);
#pragma unroll
  for (int d = 0; d < ND; ++d) *reinterpret_cast<f32x4_t*>(part + 16 * d + 4 * lg) = o[d];
  if (lg == 0) {
    part[DV] = m;
    part[DV + 1] = l;
  }
  __syncthreads();
  const int heads = min(16, rep - hg * 16);
  for (int x = threadIdx.x; x < heads * (DV / 4); x += 256) {
    const int hh = x / (DV / 4), dv = x % (DV / 4) * 4, head = g * rep + hg * 16 + hh;
    const float* from = reinterpret_cast<const float*>(lds) + hh * (DV + 4);
    float M = -INFINITY, L = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) M = fmaxf(M, from[w * (OWN / 4) + DV]);
    f32x4_t y{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = __expf(from[w * (OWN / 4) + DV] - M);
      L += f * from[w * (OWN / 4) + DV + 1];
      y += f * *reinterpret_cast<const f32x4_t*>(from + w * (OWN / 4) + dv);
    }
    if (p.nsplit > 1) {                                                     // unnormalised partials
      float* to = p.ws + ((t * p.H + head) * p.nsplit + split) * (DV + 4);
      *reinterpret_cast<f32x4_t*>(to + dv) = y;
      if (dv == 0) {
        to[DV] = M;
        to[DV + 1] = L;
      }
      continue;
    }
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    uint16_t* orow = p.out + t * p.out_ld + static_cast<int64_t>(head) * DV + dv;
    const uint16_t* grow = p.gate != nullptr ? p.gate + t * p.ld_gate + static_cast<int64_t>(head) * p.gate_dv : nullptr;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = y[i] * inv;
      if (grow != nullptr) v *= sigmoidf_(__builtin_bit_cast(float, static_cast<uint32_t>(grow[p.gate_dv > 1 ? dv + i : 0]) << 16));
      orow[i] = static_cast<uint16_t>(bf16_bits(v));
    }
  }
}

// One wave per (token, query head), or four of them: combines the splits' partials (each with its own running maximum), applies the gate. Four
// entries a lane, eight splits of a wave on their way at once, the first beside the maxima. Partials come from other XCDs' launches, some 4 us
// for a round of loads: 32 splits of 16 heads of 192 took 17 us a split after the other, 4.4 with four waves' rounds at once.
template <int WAVES>
__global__ __launch_bounds__(256) void window_pool_merge_kernel(const float* __restrict__ ws, const uint16_t* __restrict__ gate,
                                                                int64_t ld_gate, int gate_dv, uint16_t* __restrict__ out,
                                                                int64_t items, int H, int Dv, int nsplit, int64_t out_ld, float m0,
                                                                const float* __restrict__ sinks) {
  constexpr int AHEAD = 8;
  __shared__ f32x4_t sums[WAVES > 1 ? WAVES : 1][WAVES > 1 ? kWave : 1];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * (4 / WAVES) + wave / WAVES;
  if (item >= items) return;
  const int64_t t = item / H;
  const int h = static_cast<int>(item - t * H), own = wave % WAVES;
  const float* w = ws + item * nsplit * (Dv + 4);
  const int dv = 4 * lane, at = min(dv, Dv - 4);
  f32x4_t y[AHEAD];
#pragma unroll
  for (int s = 0; s < AHEAD; ++s) y[s] = *reinterpret_cast<const f32x4_t*>(w + min(own + WAVES * s, nsplit - 1) * (Dv + 4) + at);
  // lane s holds split s (at most kWave of them): its maximum and sum, then the factor that brings it to the common maximum
  const float m0h = sinks != nullptr ? sinks[h] : m0;
  const bool in = lane < nsplit;
  const float ms = in ? w[lane * (Dv + 4) + Dv] : -INFINITY, ls = in ? w[lane * (Dv + 4) + Dv + 1] : 0.0f;
  const float mm = fmaxf(m0h, wave_max(ms));
  const float f = in ? expf(ms - mm) : 0.0f;
  const float ll = wave_sum(ls * f);
  const float inv = ll > 0.0f ? 1.0f / ll : 0.0f;
  f32x4_t acc{0.0f, 0.0f, 0.0f, 0.0f};
  for (int s0 = own;; ) {
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) {
      const float fs = __shfl(f, min(s0 + WAVES * s, kWave - 1), kWave);
      if (s0 + WAVES * s < nsplit) acc += fs * y[s];
    }
    s0 += WAVES * AHEAD;
    if (s0 >= nsplit) break;
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) y[s] = *reinterpret_cast<const f32x4_t*>(w + min(s0 + WAVES * s, nsplit - 1) * (Dv + 4) + at);
  }
  if constexpr (WAVES > 1) {
    sums[own][lane] = acc;
    __syncthreads();
    if (own > 0) return;
#pragma unroll
    for (int i = 1; i < WAVES; ++i) acc += sums[i][lane];
  }
  if (dv >= Dv) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float val = acc[i] * inv;
    if (gate != nullptr)
      val *= sigmoidf_(__builtin_bit_cast(float, static_cast<uint32_t>(gate[t * ld_gate + static_cast<int64_t>(h) * gate_dv +
                                                                            (gate_dv > 1 ? dv + i : 0)]) << 16));
    out[t * out_ld + static_cast<int64_t>(h) * Dv + dv + i] = static_cast<uint16_t>(bf16_bits(val));
  }
}

// ---------------------------------------------------------------------------------------------------- prompts
// Steps that bring more than a tile of queries, on the head sizes that the models use. A wave owns 32 consecutive queries of one
// head and walks 64 keys a tile on v_mfma_f32_32x32x16_bf16: S^T = K Q^T leaves a query in each lane (its keys in 16 registers and the
// lane 32 further), and the rounded probabilities are the right-hand operand of O^T += V^T P^T as they lie. The four waves take
// up to four heads of one kv head (fewer heads: further queries), and share the K and V tile in LDS: bytes in flight per product
// are a quarter of the 16-query form above, whose waves fetch every key row for themselves.
// Tiles of tokens start at multiples of 64, so that a tile lies in one page and a thread's address is the page's plus a constant;
// pooled entries and kept first tokens are looked up row by row. SAME: the values are the first DV entries of the key rows, one tile
// serves both. Two buffers: a tile is computed while the next one's rows are on their way in registers.
// The running maximum is held in the domain of exp2 and follows every query: its largest probability is then 1, which rounding to
// bf16 leaves as it is. (Letting it lag by 2^6 saved 10 of 576 us and took the error against float64 from 2.0e-3 to 2.3e-3, at
// 64-wide heads; the 16-query form has 2.0e-3.)
// Bound by the matrix pipe and the LDS reads that feed it, about level at 32 queries a wave. Against the 16-query form on one box: 11
// prompts of 1500 tokens on average, window 1024, 16 heads over 4 of 128: 478 -> 220 us; 16 x 1024 tokens, 16 heads on latent rows of 256
// (values 192): 978 -> 195 us (342 while their rows passed through registers and 54 of them spilled); 1 x 4000 full causal, 16 over 4:
// 391 -> 122 us; 17 tokens behind 4000: 67 -> 43 us. With four query heads a kv head never slower from 17 new tokens on; with fewer see
// prompt_pays.
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((address_space(3))) unsigned char lds_u8;
constexpr int kPromptQ = 32;

// byte of 16-byte chunk ch of row `row`: rows of 256 bytes and more turn their 16 lowest chunks by the row so that 16 rows read at
// one chunk, and 4 rows x 4 chunks read transposed, meet different banks; rows of 128 bytes do so in pairs
template <int ROW_BYTES>
__device__ __forceinline__ int prompt_off(int row, int ch) {
  if constexpr (ROW_BYTES == 128) return 128 * row + 16 * (ch ^ ((((row >> 1) & 1) << 2) | ((row >> 2) & 3)));
  else return ROW_BYTES * row + 16 * (ch ^ (((row & 3) << 2) | ((row >> 2) & 3)));
}

__device__ __forceinline__ float half_max(float x) {
  const unsigned xb = __builtin_bit_cast(unsigned, x);
  const auto sw = __builtin_amdgcn_permlane32_swap(xb, xb, false, false);
  const unsigned lo = sw[0], hi = sw[1];
  return fmaxf(__builtin_bit_cast(float, lo), __builtin_bit_cast(float, hi));
}

// The 32 queries from row rw of sequence b, head h, key by key, each on the keys that it sees: for waves whose products met an
// infinity or a NaN behind a mask. Lanes c and c + 32 hold query c and half of its entries each. It starts from the kernel's arguments
// again so that nothing of it stays in registers through the kernel that ends with it.
// LATENT: the queries 16 pass .. 16 pass + 15 alone, whose rows lie in q_lds; their sums go to o_lds, rows of DV.
template <int DK, int DV, int FORM, bool LATENT = false>
__device__ __forceinline__ void prompt_redo(int b, int h, int rw, const bf16_t* q_lds = nullptr, bf16_t* o_lds = nullptr, int pass = 0) {
  typedef const __attribute__((address_space(4))) WindowMfmaParams* kernarg_t;
  kernarg_t pp = (kernarg_t)__builtin_amdgcn_kernarg_segment_ptr();
  int lane = threadIdx.x & 63;
  asm volatile("" : "+s"(pp), "+s"(b), "+s"(h), "+s"(rw), "+v"(lane));
  const auto& p = *pp;
  constexpr float kLog2e = 1.44269504088896f;
  const int c = lane & 31, half = lane >> 5, g = h / (p.H / p.G);
  const int q0 = p.cu_q[b], n = p.cu_q[b + 1] - q0, ctx = p.ctx_lens[b], row = min(rw + c, n - 1), pos = ctx + row;
  const int64_t t = q0 + row, GD = static_cast<int64_t>(p.G) * DK, GDv = static_cast<int64_t>(p.G) * DV;
  const int32_t* bt = p.block_tables + static_cast<int64_t>(b) * p.bt_stride;
  const int lo = p.chunk > 0 ? pos / p.chunk * p.chunk : max(0, pos - p.window + 1);      // first token of this query's window or chunk
  const int from = __shfl(lo, 0, kWave), w1 = ctx + min(n, rw + kPromptQ) - 1;              // of the wave's first query; last query
  const int early = p.P > 0 ? (p.chunk == 0 && w1 - p.window + 1 > 0 ? (w1 - p.window + 1) / p.P : 0) : min(p.keep_first, from);
  const float sink = p.sinks != nullptr ? p.sinks[h] : p.m0;
  constexpr int PARTS = DV > 128 ? DV / 64 : 1, ND = DV / 8 / PARTS;                      // wide rows in parts: registers
  const bf16_t* q = (LATENT ? q_lds + (c & 15) * DK : reinterpret_cast<const bf16_t*>(p.q) + (t * p.H + h) * DK) + 4 * half;
#pragma unroll 1
  for (int col = 0; col < DV; col += DV / PARTS) {
    float m = (sink < -1e30f ? -1e30f : sink) * kLog2e, l = p.sink, o[ND][4];
#pragma unroll
    for (int d = 0; d < ND; ++d) o[d][0] = o[d][1] = o[d][2] = o[d][3] = 0.0f;
#pragma unroll 1
    for (int x = 0; x < early + w1 + 1 - from; ++x) {
      const bool first = x < early, pooled = first && p.P > 0;
      const int e = first ? x : from + x - early, at = pooled ? e * p.P + p.P - 1 : e, pj = at / p.page;
      const int64_t slot = pooled ? static_cast<int64_t>(bt[pj]) * p.PP + (e - p.page * pj / p.P) : static_cast<int64_t>(bt[pj]) * p.page + at % p.page;
      const bf16_t* k = reinterpret_cast<const bf16_t*>(pooled ? p.kp + slot * GD : p.k_cache + slot * p.k_ld) + g * DK + 4 * half;
      const bf16_t* v = reinterpret_cast<const bf16_t*>(pooled ? p.vp + slot * GDv : p.v_cache + slot * p.v_ld) + g * DV + col + 4 * half;
      float s = 0.0f;
#pragma unroll 4
      for (int y = 0; y < DK; y += 8) {
        const float4 u = ld4(q + y), w = ld4(k + y);
        s = fmaf(u.x, w.x, fmaf(u.y, w.y, fmaf(u.z, w.z, fmaf(u.w, w.w, s))));
      }
      s += __shfl_xor(s, 32, kWave);
      if constexpr (FORM == kPlain) s *= p.scale;
      if constexpr (FORM == kCapped) s = p.cap * fast_tanh(s * p.cap_in);
      if constexpr (FORM == kExtended) {
        s *= p.scale * (p.key_scale != nullptr ? p.key_scale[slot * p.G + g] : 1.0f);
        if (p.dist_bias != nullptr) s += p.dist_bias[static_cast<int64_t>(h) * p.bias_len + min(max(pos - e, 0), p.bias_len - 1)];
      }
      s *= kLog2e;
      if (pooled ? at <= pos - p.window : e <= pos && (e >= lo || e < p.keep_first)) {
        const float nm = fmaxf(m, s), f = __builtin_amdgcn_exp2f(m - nm), pe = __builtin_amdgcn_exp2f(s - nm);
        const float pr = static_cast<float>(static_cast<__bf16>(pe));
        m = nm;
        l = l * f + pe;
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          const float4 u = ld4(v + 8 * d);
          o[d][0] = fmaf(pr, u.x, o[d][0] * f);
          o[d][1] = fmaf(pr, u.y, o[d][1] * f);
          o[d][2] = fmaf(pr, u.z, o[d][2] * f);
          o[d][3] = fmaf(pr, u.w, o[d][3] * f);
          if (d % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (rw + c >= n || (LATENT && (c >> 4) != pass)) continue;
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    bf16_t* orow = (LATENT ? o_lds + (c & 15) * DV : reinterpret_cast<bf16_t*>(p.out) + t * p.out_ld + static_cast<int64_t>(h) * DV) + col + 4 * half;
    const bf16_t* grow = p.gate != nullptr && (!LATENT || p.gate_dv == 1) ? reinterpret_cast<const bf16_t*>(p.gate) + t * p.ld_gate + static_cast<int64_t>(h) * p.gate_dv : nullptr;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      float y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        y[i] = o[d][i] * inv * (grow != nullptr ? sigmoidf_(ldf(grow + (p.gate_dv > 1 ? col + 8 * d + 4 * half + i : 0))) : 1.0f);
      st4(orow + 8 * d, float4{y[0], y[1], y[2], y[3]});
    }
  }
}

// DN > 0, latent attention: a wave turns its 32 queries of DN entries into rows that meet the cached ones, rotates the DK - DV entries
// behind them, and multiplies its sums by the head's value matrix before they leave, so that neither the DK entries a head that go in
// nor the DV that come out pass through memory. 16 x 1024 tokens, 16 heads of 128 + 64 on rows of 192 + 64: 201 us, where this kernel took 177,
// the two batched products around it 111 and the rotation's launch 27 (another box). A head's matrix comes in pieces of 8 KB through the wave's own part
// of the two tiles, one piece on its way while the other is multiplied; all workgroups of a head run on one XCD (with 8 sequences times
// head groups or a multiple), whose L2 holds it. A product's result rows are its matrix's columns in the order in which the next product
// takes them, so that nothing is exchanged between lanes.
template <int DK, int DV, bool SAME, int FORM, int DN = 0>
__global__ __launch_bounds__(256, DK == 64 ? 3 : 2) void prompt_attn_kernel(std::conditional_t<(DN > 0), LatentParams, WindowMfmaParams> p, int hpw,
                                                                            int tiles, int by_count) {
  constexpr int KB = DK * 2, VB = SAME ? KB : DV * 2;                       // bytes of a staged row
  constexpr int KT = kTileK * KB, VT = SAME ? 0 : kTileK * VB;
  constexpr int KCH = DK / 8, VCH = DV / 8, KN = kTileK * KCH / 256, VN = SAME ? 0 : kTileK * VCH / 256;
  constexpr int NS = DK / 16, ND = DV / 32;
  constexpr bool FIRST = DK <= 128;                                         // latent rows come without pooled blocks and kept tokens
  constexpr float kLog2e = 1.44269504088896f;
  constexpr bool DMA = !FIRST;
  static_assert(!DMA || (SAME && KB == 512 && FORM == kPlain), "rows of 512 bytes, two of them a load instruction");
  static_assert(DN == 0 || (DMA && (DK == DV || DK - DV == 64)), "own queries and outputs: latent rows, nothing or 64 entries rotated");
  constexpr int DR = DN > 0 ? DK - DV : 0, QW = DN > 0 ? DN + DR : DK;      // entries of a query's head
  __shared__ float turn_lds[DR > 0 ? 2 : 1][DR > 0 ? DR / 2 * kPromptQ : 1];                       // cosines, then sines: [frequency][query]
  __shared__ __attribute__((aligned(16))) unsigned char lds[DMA ? 16 : 2 * (KT + VT)];
  __shared__ __attribute__((aligned(1024))) unsigned char tile0[DMA ? KT : 16];
  __shared__ __attribute__((aligned(1024))) unsigned char tile1[DMA ? KT : 16];
  __shared__ __attribute__((aligned(16))) float ks_lds[FORM == kExtended ? 2 * kTileK : 4];
  __shared__ float bias_lds[FORM == kExtended ? 4 * kBiasLds : 1];
  lds_u8* const base3 = (lds_u8*)lds;
  // sequences and kv heads fastest: with a multiple of 8 of them all tiles of one run on one XCD; last queries (most keys) first
  const int by = blockIdx.x % by_count, xt = tiles - 1 - blockIdx.x / by_count;
  constexpr bool LATENT = DN > 0;                                           // one kv head, no chunks, rows without gaps: known here, not read
  const int groups = LATENT ? p.ngroups : p.G * p.ngroups, b = by / groups, gy = by % groups;
  const int g = LATENT ? 0 : gy / p.ngroups, hg = LATENT ? gy : gy % p.ngroups;
  const int q0 = p.cu_q[b], n = p.cu_q[b + 1] - q0;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, c = lane & 31, half = lane >> 5;
  const int r0 = xt * kPromptQ * (4 / hpw);
  if (r0 >= n) return;
  const int ctx = p.ctx_lens[b];
  const int h = g * (p.H / p.G) + hg * hpw + wave % hpw;
  const int rw = r0 + kPromptQ * (wave / hpw);                              // first query row of this wave
  const int i0 = ctx + r0, i1 = ctx + min(n, r0 + kPromptQ * (4 / hpw)) - 1;
  const bool live = rw < n;
  const int w0 = ctx + rw, w1 = ctx + min(n, rw + kPromptQ) - 1;            // positions of this wave's first and last query
  const int row = min(rw + c, n - 1), pos = ctx + row;
  const int64_t t = q0 + row;
  const int page = p.page, P = LATENT ? 0 : p.P, W = p.window, chunk = LATENT ? 0 : p.chunk, keep = LATENT ? 0 : p.keep_first;
  const int cstart = chunk > 0 ? (pos / chunk) * chunk : 0;
  const int32_t* bt = p.block_tables + static_cast<int64_t>(b) * p.bt_stride;
  const int64_t GD = static_cast<int64_t>(p.G) * DK, GDv = static_cast<int64_t>(p.G) * DV, k_ld = LATENT ? DK : p.k_ld;

  bf16x8_t qf[NS];
  lds_u8* const slot0 = (lds_u8*)tile0 + 8192 * wave;                       // the wave's own parts of the tiles
  lds_u8* const slot1 = (lds_u8*)tile1 + 8192 * wave;
  const int tq = (lane & 15) >> 2, tp = lane & 3, gi = lane >> 4;           // transposed reads: 16 lanes read 4 rows x 16 columns
  auto landed = [&](auto later) __attribute__((always_inline)) {            // own pieces, but for the `later` youngest loads
    constexpr int n = decltype(later)::value;
    __builtin_amdgcn_s_waitcnt(n | 0x0f70);
    asm volatile("" ::: "memory");
  };
  auto reads_done = [&]() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);                                     // lgkmcnt(0)
    asm volatile("" ::: "memory");
  };
  auto cast8 = [](const f32x16_t& x, int from) __attribute__((always_inline)) {
    bf16x8_t y;
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = static_cast<__bf16>(x[from + i]);
    return y;
  };
  // a sum of rounded products, as the launch that rotates queries by itself forms it (no product goes into the addition unrounded)
  auto rounded_sum = [](float x, float y) __attribute__((always_inline)) {
    asm volatile("" : "+v"(x), "+v"(y));
    return x + y;
  };
  // the lane's number, unknown to the compiler: what is made of it is not kept in registers from here to there
  auto lane_here = [&]() __attribute__((always_inline)) {
    int x = lane;
    asm volatile("" : "+v"(x));
    return x;
  };
  // The same of the arguments and of what this workgroup has to do: the code in front of the tile loop and behind it starts from them again. Kept
  // through the loop they left it too few registers to read four fragments ahead (17 or 1024 tokens behind 16000, 16 heads, us: batched products
  // 571 / 652, this launch 634 / 711 with them kept, 550 / 621 without).
  struct LatentArgs { LatentParams p; int hpw, tiles, by_count; };
  typedef const __attribute__((address_space(4))) LatentArgs* args_t;
  struct Own { args_t a; int h, rw, q0, n; };
  auto again = [&]() __attribute__((always_inline)) {
    args_t a = (args_t)__builtin_amdgcn_kernarg_segment_ptr();
    int block = blockIdx.x;
    asm volatile("" : "+s"(a), "+s"(block));
    const int by = block % a->by_count, b = by / a->p.ngroups, q0 = a->p.cu_q[b];
    return Own{a, by % a->p.ngroups * 4 + wave, (a->tiles - 1 - block / a->by_count) * kPromptQ, q0, a->p.cu_q[b + 1] - q0};
  };
  // rows of the key matrix, 16 a piece of 512-byte rows (of which a latent of 192 fills 384)
  auto uk_piece = [&](const Own& own, int k, lds_u8* at, int ln) __attribute__((always_inline)) {
    if constexpr (DN > 0) {
      const char* from = reinterpret_cast<const char*>(own.a->p.uk + (static_cast<int64_t>(own.h) * DN + 16 * k) * DV);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int r = 2 * i + (ln >> 5), ch = (ln & 31) ^ (((r & 3) << 2) | ((r >> 2) & 3));
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from + static_cast<uint32_t>(r * 2 * DV + 16 * min(ch, DV / 8 - 1))),
                                         (__attribute__((address_space(3))) void*)(at + 1024 * i), 16, 0, 0);
      }
    }
  };
  // qf = [q_n W_uk | rotated q_r]
  auto absorb = [&](auto beside) __attribute__((always_inline)) {
    if constexpr (DN > 0) {
      constexpr int NP = DN / 16;
      const Own own = again();
      const int ln = lane_here(), half = ln >> 5, c = ln & 31, tq = (ln & 15) >> 2, tp = ln & 3, gi = ln >> 4;
      uk_piece(own, 0, slot0, ln);
      uk_piece(own, 1, slot1, ln);
      const uint16_t* qrow = own.a->p.q + (static_cast<int64_t>(own.q0 + min(own.rw + c, own.n - 1)) * own.a->p.H + own.h) * QW + 8 * half;
      bf16x8_t raw[NP];
#pragma unroll
      for (int k = 0; k < NP; ++k) raw[k] = *reinterpret_cast<const bf16x8_t*>(qrow + 16 * k);
#pragma unroll
      for (int x = 0; x < DR / 16; ++x) qf[DV / 16 + x] = *reinterpret_cast<const bf16x8_t*>(qrow + DN + 16 * x);
      beside();
#pragma unroll
      for (int k = 0; k < NP; ++k) asm volatile("" ::"v"(raw[k]));
      f32x16_t acc[ND];
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] = 0.0f;
      // of 16 columns, fours 1 and 2 change places: a lane's results are then entries 8 half .. 8 half + 7 of two steps of K Q^T
      int addr[2][ND < 4 ? ND : 4];
#pragma unroll
      for (int second = 0; second < 2; ++second)
#pragma unroll
        for (int d = 0; d < 4; ++d)
          addr[second][d] = prompt_off<512>(8 * (gi >> 1) + 4 * second + tq, 4 * d + 2 * (gi & 1) + (tp & 1)) + 8 * (tp >> 1);
      auto multiply = [&](int k, const lds_u8* at) __attribute__((always_inline)) {
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          const bf16x4v_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(at + addr[0][d % 4] + 256 * (d / 4)));
          const bf16x4v_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(at + addr[1][d % 4] + 256 * (d / 4)));
          acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), raw[k], acc[d], 0, 0, 0);
          if (d % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
      };
#pragma unroll
      for (int k = 0; k < NP; k += 2) {
        landed(std::integral_constant<int, 8>{});
        multiply(k, slot0);
        reads_done();
        if (k + 2 < NP) {
          uk_piece(own, k + 2, slot0, ln);
          landed(std::integral_constant<int, 8>{});
        } else {
          landed(std::integral_constant<int, 0>{});
        }
        multiply(k + 1, slot1);
        reads_done();
        if (k + 3 < NP) uk_piece(own, k + 3, slot1, ln);
      }
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        qf[2 * d] = cast8(acc[d], 0);
        qf[2 * d + 1] = cast8(acc[d], 8);
      }
      if constexpr (DR > 0) {                                               // pairs (i, i + 32): a lane holds both
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          bf16x8_t &a = qf[DV / 16 + x], &z = qf[DV / 16 + 2 + x];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int at = (16 * x + 8 * half + i) * kPromptQ + c;
            const float co = turn_lds[0][at], si = turn_lds[1][at], u = static_cast<float>(a[i]), v = static_cast<float>(z[i]);
            a[i] = static_cast<__bf16>(rounded_sum(u * co, -(v * si)));
            z[i] = static_cast<__bf16>(rounded_sum(v * co, u * si));
          }
        }
      }
    }
  };
  // the wave's outputs from its sums, which lie as the value matrix takes them; pass >= 0: those of 16 queries
  auto leave = [&](const bf16x8_t* of, int pass) __attribute__((always_inline)) {
    if constexpr (DN > 0) {
      constexpr int UB = 2 * DN, UN = UB * 32 / 1024, NE = DN / 32;
      const Own own = again();
      const auto& p = own.a->p;
      const int ln = lane_here(), half = ln >> 5, c = ln & 31, tq = (ln & 15) >> 2, tp = ln & 3, gi = ln >> 4;
      auto uv_piece = [&](int k, lds_u8* at) __attribute__((always_inline)) {      // 32 rows
        const char* from = reinterpret_cast<const char*>(p.uv + (static_cast<int64_t>(own.h) * DV + 32 * k) * DN);
#pragma unroll
        for (int i = 0; i < UN; ++i) {
          const int r = (1024 / UB) * i + ln / (UB / 16), pc = ln % (UB / 16);
          const int ch = UB == 128 ? pc ^ ((((r >> 1) & 1) << 2) | ((r >> 2) & 3)) : pc ^ (((r & 3) << 2) | ((r >> 2) & 3));
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from + static_cast<uint32_t>(r * UB + 16 * ch)),
                                           (__attribute__((address_space(3))) void*)(at + 1024 * i), 16, 0, 0);
        }
      };
      uv_piece(0, slot0);
      uv_piece(1, slot1);
      int addr[2][NE];
#pragma unroll
      for (int second = 0; second < 2; ++second)
#pragma unroll
        for (int e = 0; e < NE; ++e)
          addr[second][e] = prompt_off<UB>(8 * second + 4 * (gi >> 1) + tq, 4 * e + 2 * (gi & 1) + (tp >> 1)) + 8 * (tp & 1);
      f32x16_t y[NE];
#pragma unroll
      for (int e = 0; e < NE; ++e)
#pragma unroll
        for (int i = 0; i < 16; ++i) y[e][i] = 0.0f;
      auto multiply = [&](int k, const lds_u8* at) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
#pragma unroll
          for (int e = 0; e < NE; ++e) {
            const bf16x4v_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(at + UB * 16 * x + addr[0][e]));
            const bf16x4v_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(at + UB * 16 * x + addr[1][e]));
            y[e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), of[2 * k + x], y[e], 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      };
#pragma unroll
      for (int k = 0; k < ND; k += 2) {
        landed(std::integral_constant<int, UN>{});
        multiply(k, slot0);
        reads_done();
        if (k + 2 < ND) {
          uv_piece(k + 2, slot0);
          landed(std::integral_constant<int, UN>{});
        } else {
          landed(std::integral_constant<int, 0>{});
        }
        multiply(k + 1, slot1);
        reads_done();
        if (k + 3 < ND) uv_piece(k + 3, slot1);
      }
      if (own.rw + c >= own.n || (pass >= 0 && (c >> 4) != pass)) return;
      const int64_t t = own.q0 + own.rw + c;
      bf16_t* orow = reinterpret_cast<bf16_t*>(p.out) + t * p.out_ld + static_cast<int64_t>(own.h) * DN + 4 * half;
      const bool gated = p.gate != nullptr && p.gate_dv != 1;
      const bf16_t* grow = reinterpret_cast<const bf16_t*>(p.gate) + t * p.ld_gate + static_cast<int64_t>(own.h) * DN + 4 * half;
#pragma unroll
      for (int e = 0; e < NE; ++e)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          float4 v{y[e][4 * x], y[e][4 * x + 1], y[e][4 * x + 2], y[e][4 * x + 3]};
          if (gated) {
            const float4 gv = ld4(grow + 32 * e + 8 * x);
            v = float4{v.x * sigmoidf_(gv.x), v.y * sigmoidf_(gv.y), v.z * sigmoidf_(gv.z), v.w * sigmoidf_(gv.w)};
          }
          st4(orow + 32 * e + 8 * x, v);
        }
    }
  };
  if constexpr (DN > 0) {
    absorb([&]() __attribute__((always_inline)) {
      if constexpr (DR > 0) {                                               // (the four waves have the same queries)
#pragma unroll 1
        for (int f = threadIdx.x >> 5; f < DR / 2; f += 8) {
          float si, co;
          sincosf(static_cast<float>(pos) * p.inv_freq[f], &si, &co);
          turn_lds[0][f * kPromptQ + c] = co;
          turn_lds[1][f * kPromptQ + c] = si;
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      }
    });
    asm volatile("s_barrier" ::: "memory");                                 // the tiles are everyone's again
  } else {
    const uint16_t* qrow = p.q + (t * p.H + h) * DK + 8 * half;
#pragma unroll
    for (int s = 0; s < NS; ++s) qf[s] = *reinterpret_cast<const bf16x8_t*>(qrow + 16 * s);
#pragma unroll
    for (int s = 0; s < NS; ++s) asm volatile("" ::"v"(qf[s]));            // the loads end here, not at a wait inside the tile loop
  }
  const int jlo = (chunk > 0 ? (i0 / chunk) * chunk : max(0, i0 - W + 1)) & ~(kTileK - 1);
  const int nbmax = P > 0 ? ((chunk == 0 && i1 - W + 1 > 0) ? (i1 - W + 1) / P : 0) : min(keep, jlo);
  const int npt = FIRST ? (nbmax + kTileK - 1) / kTileK : 0, ntiles = npt + (i1 - jlo) / kTileK + 1;

  // staging: chunk tid % KCH of rows tid / KCH + (256 / KCH) i
  const int k_ch = threadIdx.x % KCH, k_r = threadIdx.x / KCH, v_ch = threadIdx.x % VCH, v_r = threadIdx.x / VCH;
  u32x4_t kreg[KN], vreg[SAME ? 1 : VN];
  float ksreg = 1.0f;
  const bool keyed = FORM == kExtended && p.key_scale != nullptr && threadIdx.x < kTileK;
  auto slot_of = [&](int e) __attribute__((always_inline)) {                // row of an entry of the first phase
    const int ec = min(e, nbmax - 1);
    if (P > 0) {
      const int pj = fdiv(ec * P + P - 1, page, p.m_page);
      return static_cast<int64_t>(bt[pj]) * p.PP + (ec - fdiv(page * pj, P, p.m_P));
    }
    const int pj = fdiv(ec, page, p.m_page);
    return static_cast<int64_t>(bt[pj]) * page + (ec - pj * page);
  };
  auto load = [&](int tile) __attribute__((always_inline)) {
    if (FIRST && tile < npt) {
      const uint16_t* kb = (P > 0 ? p.kp : p.k_cache) + g * DK + 8 * k_ch;
      const uint16_t* vb = (P > 0 ? p.vp : p.v_cache) + g * DV + 8 * v_ch;
      const int64_t kld = P > 0 ? GD : p.k_ld, vld = P > 0 ? GDv : p.v_ld;
#pragma unroll
      for (int x = 0; x < KN; ++x)
        kreg[x] = *reinterpret_cast<const u32x4_t*>(kb + slot_of(tile * kTileK + k_r + 256 / KCH * x) * kld);
#pragma unroll
      for (int x = 0; x < VN; ++x)
        vreg[x] = *reinterpret_cast<const u32x4_t*>(vb + slot_of(tile * kTileK + v_r + 256 / VCH * x) * vld);
      if (keyed) ksreg = p.key_scale[slot_of(tile * kTileK + threadIdx.x) * p.G + g];
    } else {
      const int e0 = jlo + (tile - npt) * kTileK, pj = fdiv(e0, page, p.m_page), last = i1 - e0;
      const int64_t slot = static_cast<int64_t>(bt[pj]) * page + (e0 - pj * page);
      const uint16_t* kb = p.k_cache + slot * p.k_ld + g * DK;
      const uint16_t* vb = p.v_cache + slot * p.v_ld + g * DV;
#pragma unroll
      for (int x = 0; x < KN; ++x)                                          // rows past the last query's repeat its row: finite values
        kreg[x] = *reinterpret_cast<const u32x4_t*>(kb + static_cast<uint32_t>(min(k_r + 256 / KCH * x, last)) * static_cast<uint32_t>(p.k_ld) + 8 * k_ch);
#pragma unroll
      for (int x = 0; x < VN; ++x)
        vreg[x] = *reinterpret_cast<const u32x4_t*>(vb + static_cast<uint32_t>(min(v_r + 256 / VCH * x, last)) * static_cast<uint32_t>(p.v_ld) + 8 * v_ch);
      if (keyed) ksreg = p.key_scale[(slot + min(static_cast<int>(threadIdx.x), last)) * p.G + g];
    }
  };
  auto store = [&](int buf) __attribute__((always_inline)) {
    unsigned char* kt = lds + buf * (KT + VT);
#pragma unroll
    for (int x = 0; x < KN; ++x) *reinterpret_cast<u32x4_t*>(kt + prompt_off<KB>(k_r + 256 / KCH * x, k_ch)) = kreg[x];
#pragma unroll
    for (int x = 0; x < VN; ++x) *reinterpret_cast<u32x4_t*>(kt + KT + prompt_off<VB>(v_r + 256 / VCH * x, v_ch)) = vreg[x];
    if (FORM == kExtended && threadIdx.x < kTileK) ks_lds[buf * kTileK + threadIdx.x] = ksreg;
  };
  const float* bias_h = nullptr;
  bool bias_cached = false;
  if constexpr (FORM == kExtended) {
    if (p.dist_bias != nullptr) {
      bias_h = p.dist_bias + static_cast<int64_t>(h) * p.bias_len;
      bias_cached = p.bias_len <= kBiasLds;
      if (bias_cached)
        for (int x = lane; x < p.bias_len; x += kWave) bias_lds[wave * kBiasLds + x] = bias_h[x];     // read by this wave alone
    }
  }

  // LDS addresses inside a buffer: rows of K (lane = key), V transposed
  // (chunks 16 further lie 256 bytes further: a turn touches the four lowest bits)
  constexpr int NKA = NS < 8 ? NS : 8, NVA = ND < 4 ? ND : 4;
  int kaddr[NKA], vaddr[2][NVA];
#pragma unroll
  for (int x = 0; x < NKA; ++x) kaddr[x] = prompt_off<KB>(c, 2 * x + half);
#pragma unroll
  for (int second = 0; second < 2; ++second)
#pragma unroll
    for (int d = 0; d < NVA; ++d)
      vaddr[second][d] = (SAME ? 0 : KT) + prompt_off<VB>(8 * second + 4 * (gi >> 1) + tq, 4 * d + 2 * (gi & 1) + (tp >> 1)) + 8 * (tp & 1);

  f32x16_t o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.0f;
  const float cs = FORM == kPlain ? p.scale * kLog2e : kLog2e;              // from what the products leave to the exponent of 2
  // (a sink of -infinity counts nothing: a start far below any score, since a query may not see its first tiles)
  const float sink = p.sinks != nullptr ? p.sinks[h] : p.m0;
  float m = (sink < -1e30f ? -1e30f : sink) * kLog2e, l = half == 0 ? p.sink : 0.0f;
  // tiles that hold nothing for this wave's queries, and tiles of tokens that all of them see whole
  auto skipped = [&](int phase, int e0) __attribute__((always_inline)) {
    if (phase == 0) return P > 0 && e0 * P + P - 1 > w1 - W;
    return e0 > w1 || (e0 >= keep && (chunk > 0 ? e0 + kTileK - 1 < (w0 / chunk) * chunk : w0 - (e0 + kTileK - 1) >= W));
  };
  auto seen_whole = [&](int e0) __attribute__((always_inline)) {
    return e0 + kTileK - 1 <= w0 && (chunk > 0 ? e0 >= w1 - w1 % chunk : w1 - e0 < W);
  };

  auto compute = [&](int tile, int buf, lds_u8* kt) __attribute__((always_inline)) {
    const int phase = FIRST && tile < npt ? 0 : 1;
    const int e0 = phase == 0 ? tile * kTileK : jlo + (tile - npt) * kTileK;
    const int e_end = phase == 0 ? nbmax : i1 + 1;
    if (!live || skipped(phase, e0)) return;
    const bool whole = phase == 1 && seen_whole(e0);
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      f32x16_t s;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
      for (int x = 0; x < NS; ++x) {
        const bf16x8_t ka = *reinterpret_cast<const __attribute__((address_space(3))) bf16x8_t*>(kt + kaddr[x % NKA] + (KB * 32 * sub + 256 * (x / NKA)));
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka, qf[x], s, 0, 0, 0);
        if (DK == 256 && x % 4 == 3) __builtin_amdgcn_sched_barrier(0);     // fragments of four steps at a time: more of them spill
      }
      const int ks0 = e0 + 32 * sub;
      if constexpr (FORM == kCapped) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = p.cap * fast_tanh(s[i] * p.cap_in);
      }
      if constexpr (FORM == kExtended) {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const f32x4_t ks = *reinterpret_cast<const f32x4_t*>(ks_lds + buf * kTileK + 32 * sub + 8 * x + 4 * half);
#pragma unroll
          for (int i = 0; i < 4; ++i) s[4 * x + i] *= ks[i] * p.scale;
        }
        if (bias_h != nullptr) {
          const float* table = bias_cached ? bias_lds + wave * kBiasLds : bias_h;
          const int top = p.bias_len - 1;
          if (w0 - (ks0 + 31) >= top) {                                     // all of the tile at the last bias
            const float far = table[top];
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] += far;
          } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const int dist = min(max(pos - (ks0 + (i & 3) + 8 * (i >> 2) + 4 * half), 0), top);
              s[i] += table[dist];
            }
          }
        }
      }
      if (!whole) {
        if constexpr (LATENT) asm volatile("");                             // a branch: most tiles have no mask
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int ke = ks0 + (i & 3) + 8 * (i >> 2) + 4 * half;
          bool vis = ke < e_end;
          if (phase == 0) vis = vis && (P == 0 || ke * P + P - 1 <= pos - W);
          else vis = vis && ke <= pos && ((chunk > 0 ? ke >= cstart : pos - ke < W) || ke < keep);
          s[i] = vis ? s[i] : -INFINITY;
        }
      }
      float mx = s[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
      mx = half_max(mx) * cs;
      if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {
        const float nm = fmaxf(m, mx), f = __builtin_amdgcn_exp2f(m - nm);
        m = nm;
        l *= f;
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[d][i] *= f;
      }
      bf16x8_t pf[2];
      float sum = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float e = __builtin_amdgcn_exp2f(fmaf(s[i], cs, -m));
        sum += e;
        pf[i >> 3][i & 7] = static_cast<__bf16>(e);
      }
      l += sum;
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        if (DK == 256) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          const lds_u8* v = kt + VB * (32 * sub + 16 * x);
          const bf16x4v_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(v + vaddr[0][d % NVA] + 256 * (d / NVA)));
          const bf16x4v_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(v + vaddr[1][d % NVA] + 256 * (d / NVA)));
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), pf[x], o[d], 0, 0, 0);
          if (DK == 256 && d % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };

  if constexpr (DMA) {
    // Latent rows go straight from memory into the tile, whose buffers are arrays of their own so that the compiler sees which of
    // them a read has to wait for; held in registers on the way they cost 32 of the wave's 256, and accumulators spilled.
    const int d_r = 2 * wave + half;                                        // row of piece `wave`; piece wave + 4 i: 8 i further
    auto request = [&](int tile, lds_u8* at) __attribute__((always_inline)) {
      const int e0 = jlo + tile * kTileK, pj = fdiv(e0, page, p.m_page), last = i1 - e0;
      const int64_t slot = static_cast<int64_t>(bt[pj]) * page + (e0 - pj * page);
      const char* kb = reinterpret_cast<const char*>(p.k_cache + slot * k_ld + g * DK);
#pragma unroll
      for (int i = 0; i < KT / 4096; ++i) {
        const int r = 8 * i + d_r, ch = (lane & 31) ^ (((r & 3) << 2) | ((r >> 2) & 3));
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)(kb + static_cast<uint32_t>(min(r, last)) * static_cast<uint32_t>(2 * k_ld) + 16 * ch),
            (__attribute__((address_space(3))) void*)(at + 1024 * (wave + 4 * i)), 16, 0, 0);
      }
    };
    auto turn = [&]() __attribute__((always_inline)) {
      __builtin_amdgcn_s_waitcnt(0x0070);                                   // own pieces landed, own reads done; then everyone's
      asm volatile("s_barrier" ::: "memory");
    };
    request(0, (lds_u8*)tile0);
    turn();
    for (int tile = 0;;) {
      if (tile + 1 < ntiles) request(tile + 1, (lds_u8*)tile1);
      compute(tile, 0, (lds_u8*)tile0);
      turn();
      if (++tile >= ntiles) break;
      if (tile + 1 < ntiles) request(tile + 1, (lds_u8*)tile0);
      compute(tile, 1, (lds_u8*)tile1);
      turn();
      if (++tile >= ntiles) break;
    }
  } else {
    load(0);
    store(0);
    __syncthreads();
    if (ntiles > 1) load(1);
    for (int tile = 0; tile < ntiles; ++tile) {
      compute(tile, tile & 1, base3 + (tile & 1) * (KT + VT));
      if (tile + 1 < ntiles) store((tile + 1) & 1);
      if (tile + 2 < ntiles) load(tile + 2);
      __syncthreads();
    }
  }
  if (!live) return;
  // A probability of zero does not keep an infinity or a NaN of a value row out of the products. Where an output is not finite, the value
  // rows of the tiles that had a mask are looked at, and if one of them is the cause the wave's queries are done again (prompt_redo).
  float odd = 0.0f;
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) odd = fmaf(o[d][i], 0.0f, odd);
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(odd != 0.0f) != 0, 0)) {
    auto row_of = [&](int e, bool first) __attribute__((always_inline)) {
      if (first) return slot_of(e);
      const int pj = fdiv(e, page, p.m_page);
      return static_cast<int64_t>(bt[pj]) * page + (e - pj * page);
    };
    const uint16_t *kp = P > 0 ? p.kp : p.k_cache, *vp = P > 0 ? p.vp : p.v_cache;
    const int64_t kp_ld = P > 0 ? GD : p.k_ld, vp_ld = P > 0 ? GDv : p.v_ld;
    bool bad = false;
#pragma unroll 1
    for (int tile = 0; tile < ntiles; ++tile) {
      const bool first = tile < npt;
      const int e0 = first ? tile * kTileK : jlo + (tile - npt) * kTileK;
      if (skipped(first ? 0 : 1, e0) || (!first && seen_whole(e0))) continue;
      const int e = min(e0 + lane, first ? nbmax - 1 : i1);
      const uint16_t* v = first ? vp + row_of(e, true) * vp_ld + g * DV : p.v_cache + row_of(e, false) * p.v_ld + g * DV;
#pragma unroll 1
      for (int x = 0; x < DV; x += 2) {
        const uint32_t u = *reinterpret_cast<const uint32_t*>(v + x);
        bad = bad || (u & 0x7f80u) == 0x7f80u || (u & 0x7f800000u) == 0x7f800000u;
      }
    }
    if (__builtin_amdgcn_ballot_w64(bad) != 0) {
      if constexpr (DN == 0) {
        prompt_redo<DK, DV, FORM>(b, __builtin_amdgcn_readfirstlane(h), __builtin_amdgcn_readfirstlane(rw));
        return;
      } else {
        bf16_t *q_at = reinterpret_cast<bf16_t*>(tile0 + 8192 * wave), *o_at = reinterpret_cast<bf16_t*>(tile1 + 8192 * wave);
#pragma unroll 1
        for (int pass = 0; pass < 2; ++pass) {
          absorb([] {});
          if ((c >> 4) == pass) {
#pragma unroll
            for (int s = 0; s < NS; ++s) *reinterpret_cast<bf16x8_t*>(q_at + (c & 15) * DK + 16 * s + 8 * half) = qf[s];
          }
          reads_done();
          prompt_redo<DK, DV, FORM, true>(b, __builtin_amdgcn_readfirstlane(h), __builtin_amdgcn_readfirstlane(rw), q_at, o_at, pass);
          reads_done();
          bf16x8_t of[2 * ND];
#pragma unroll
          for (int d = 0; d < 2 * ND; ++d) {
            const uint2 lo = *reinterpret_cast<const uint2*>(o_at + (c & 15) * DV + 16 * d + 4 * half);
            const uint2 hi = *reinterpret_cast<const uint2*>(o_at + (c & 15) * DV + 16 * d + 8 + 4 * half);
            of[d] = __builtin_bit_cast(bf16x8_t, uint4{lo.x, lo.y, hi.x, hi.y});
          }
          reads_done();
          leave(of, pass);
        }
        return;
      }
    }
  }
  const float total = l + __shfl_xor(l, 32, kWave);
  const float inv = total > 0.0f ? 1.0f / total : 0.0f;
  if constexpr (DN > 0) {
    const Own own = again();
    const int c = lane_here() & 31;
    const bf16_t* gate = reinterpret_cast<const bf16_t*>(own.a->p.gate);
    const int64_t t = own.q0 + min(own.rw + c, own.n - 1);
    const float gate1 = gate != nullptr && own.a->p.gate_dv == 1 ? sigmoidf_(ldf(gate + t * own.a->p.ld_gate + own.h)) : 1.0f;
    bf16x8_t of[2 * ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) {
#pragma unroll
      for (int i = 0; i < 16; ++i) o[d][i] = o[d][i] * inv * gate1;         // (the order of the outputs without matrices)
      of[2 * d] = cast8(o[d], 0);
      of[2 * d + 1] = cast8(o[d], 8);
      __builtin_amdgcn_sched_barrier(0);
    }
    leave(of, -1);
    return;
  }
  if (rw + c >= n) return;
  uint16_t* orow = p.out + t * p.out_ld + static_cast<int64_t>(h) * DV + 4 * half;
  const uint16_t* grow = p.gate != nullptr ? p.gate + t * p.ld_gate + static_cast<int64_t>(h) * p.gate_dv : nullptr;
  const float gate1 = grow != nullptr && p.gate_dv == 1 ? sigmoidf_(ldf(reinterpret_cast<const bf16_t*>(grow))) : 1.0f;
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      float4 y{o[d][4 * x] * inv, o[d][4 * x + 1] * inv, o[d][4 * x + 2] * inv, o[d][4 * x + 3] * inv};
      if (grow != nullptr) {
        if (p.gate_dv == 1) {
          y = float4{y.x * gate1, y.y * gate1, y.z * gate1, y.w * gate1};
        } else {
          const float4 gv = ld4(reinterpret_cast<const bf16_t*>(grow) + 32 * d + 8 * x + 4 * half);
          y = float4{y.x * sigmoidf_(gv.x), y.y * sigmoidf_(gv.y), y.z * sigmoidf_(gv.z), y.w * sigmoidf_(gv.w)};
        }
      }
      st4(reinterpret_cast<bf16_t*>(orow) + 32 * d + 8 * x, y);
    }
}

// Whether 32 queries a wave pay. A workgroup takes fewer than four heads of a kv head as so many more queries of each, so a launch
// that leaves most of the chip idle has fewer workgroups, with a longer chain of tiles each, than one with 16 queries a wave, whose
// spare waves cost nothing there. With a multiple of four heads both have waves to fill. us, 16 / 32 queries: 100 tokens, 8 heads of 64
// over 8 8.4 / 13.2, of 128 10.0 / 15.6, behind 1000 tokens 31.4 / 37.3; 16 over 8 9.1 / 10.0, but behind 1000 36.0 / 34.2; 6 over 2
// 9.8 / 13.2; 16 x 500 tokens, 8 over 8 82.7 / 23.8. `keys`: what a workgroup of 16 queries passes, from the table's width. The lines
// lie where the two cross in 1450 launches of 1 to 16 sequences of 17 to 1000 tokens behind 0 to 3000: the choice is within 14 % of
// the better one, 0.6 % off it on average.
static bool prompt_pays(const WindowMfmaParams& p, int64_t T, int B, int max_new) {
  const int rep = p.H / p.G;
  if (rep % 4 == 0 || rep == 6 || p.D > 128) return true;
  int64_t keys = static_cast<int64_t>(p.bt_stride) * p.page, units = static_cast<int64_t>(B) * ((max_new + kTileQ - 1) / kTileQ);
  if (T > 0) units = std::min<int64_t>(units, (T + static_cast<int64_t>(B) * (kTileQ - 1)) / kTileQ);
  const int64_t pooled = p.P > 0 ? keys / p.P : 0;
  keys = std::min<int64_t>(keys, (p.chunk > 0 ? p.chunk : p.window) + static_cast<int64_t>(kTileQ) + p.keep_first) + pooled;
  const bool few = max_new <= 2 * kPromptQ;                                 // at most two of the four waves have queries
  const int64_t most = rep == 1 ? (few ? 768 : 2048) : rep == 2 ? (few ? 512 : 768) : (few ? 0 : 256);
  const int64_t volume = rep == 1 ? (few ? 8 : 24) : (few ? 4 : 8);
  return keys > most || units * p.G * keys * p.D > volume << 20;
}

// The head sizes and forms that prompt_attn_kernel is built for; false: the launch belongs to window_pool_mfma_kernel. It also
// needs pages of whole tiles, a positive scale (the maximum is taken before it is applied), and rows that allow 8-byte accesses of
// gate and output.
static bool prompt_launch(const WindowMfmaParams& p, int form, int64_t T, int B, int max_new, bool forced, hipStream_t s) {
  auto at = [](const void* q, uintptr_t a) { return reinterpret_cast<uintptr_t>(q) % a == 0; };
  if (p.D > 128 && (p.P > 0 || p.keep_first > 0)) return false;
  if (max_new <= kTileQ || p.page % kTileK != 0 || !(p.scale > 0.0f) || !at(p.q, 16) || !at(p.out, 8) || p.out_ld % 4 != 0 ||
      (p.P > 0 && (!at(p.kp, 16) || !at(p.vp, 16))) ||
      (p.gate != nullptr && p.gate_dv > 1 && (!at(p.gate, 8) || p.ld_gate % 4 != 0)))
    return false;
  if (!forced && !prompt_pays(p, T, B, max_new)) return false;
  const bool same = p.P == 0 && (p.G == 1 || p.D == p.Dv) && p.k_cache == p.v_cache && p.k_ld == p.v_ld;
  const int rep = p.H / p.G, hpw = rep % 4 == 0 ? 4 : (rep % 2 == 0 ? 2 : 1);
  WindowMfmaParams q = p;
  q.ngroups = rep / hpw;
  const int rows = kPromptQ * (4 / hpw), tiles = (max_new + rows - 1) / rows, by = B * p.G * q.ngroups;
  if (static_cast<int64_t>(tiles) * by >= (1ll << 31)) return false;
  const dim3 grid(static_cast<unsigned>(tiles) * by), block(256);
#define LVMIX_PROMPT(DK, DV, SAME, FORM)                                                              \
  if (p.D == DK && p.Dv == DV && same == SAME && form == FORM) {                                      \
    prompt_attn_kernel<DK, DV, SAME, FORM><<<grid, block, 0, s>>>(q, hpw, tiles, by);                 \
    return true;                                                                                      \
  }
  LVMIX_PROMPT(64, 64, false, kPlain)
  LVMIX_PROMPT(64, 64, false, kCapped)
  LVMIX_PROMPT(64, 64, false, kExtended)
  LVMIX_PROMPT(128, 128, false, kPlain)
  LVMIX_PROMPT(128, 128, false, kCapped)
  LVMIX_PROMPT(128, 128, false, kExtended)
  LVMIX_PROMPT(128, 128, true, kPlain)
  LVMIX_PROMPT(128, 128, true, kExtended)
  LVMIX_PROMPT(256, 192, true, kPlain)
  LVMIX_PROMPT(256, 256, true, kPlain)
#undef LVMIX_PROMPT
  return false;
}

// The head sizes that decode_pool_kernel is built for; false: the launch belongs to window_pool_mfma_kernel. Rows of q, caches and workspace
// are read 16 bytes at a time. (mix_ops.decode_heads restates this for the count of splits.)
static bool decode_launch(const WindowMfmaParams& p, int form, int B, hipStream_t s) {
  auto at = [](const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 == 0; };
  if (form != kPlain || !at(p.q) || !at(p.ws) || (p.P > 0 && (!at(p.kp) || !at(p.vp)))) return false;
  const bool same = p.P == 0 && (p.G == 1 || p.D == p.Dv) && p.k_cache == p.v_cache && p.k_ld == p.v_ld;
  WindowMfmaParams q = p;
  q.ngroups = (p.H / p.G + 15) / 16;
  const dim3 grid(p.nsplit, p.G * q.ngroups, B), block(256);
  if (p.D == 64 && p.Dv == 64 && !same) decode_pool_kernel<64, 64, false><<<grid, block, 0, s>>>(q);
  else if (p.D == 64 && p.Dv == 64) decode_pool_kernel<64, 64, true><<<grid, block, 0, s>>>(q);
  else if (p.D == 128 && p.Dv == 128 && !same) decode_pool_kernel<128, 128, false><<<grid, block, 0, s>>>(q);
  else if (p.D == 128 && p.Dv == 128) decode_pool_kernel<128, 128, true><<<grid, block, 0, s>>>(q);
  else if (p.D == 256 && p.Dv == 192 && same) decode_pool_kernel<256, 192, true><<<grid, block, 0, s>>>(q);
  else if (p.D == 256 && p.Dv == 256 && same) decode_pool_kernel<256, 256, true><<<grid, block, 0, s>>>(q);
  else return false;
  return true;
}

}  // namespace lvmix

using namespace lvmix;

static uint32_t magic(int d) { return d <= 1 ? 0xffffffffu : static_cast<uint32_t>((1ull << 32) / static_cast<uint64_t>(d)); }

extern "C" int lv_window_pool_attn_mfma(const void* q, const void* k_cache, const void* v_cache, const void* kp,
                                        const void* vp, const void* gate, int64_t ld_gate, void* out, const int32_t* cu_q,
                                        const int32_t* ctx_lens, const int32_t* block_tables, int bt_stride, int B,
                                        int max_new_tokens, int H, int G, int D, int Dv, int page, int window, int P,
                                        float scale, int has_sink, int nsplit, void* workspace, int64_t T, int64_t k_ld,
                                        int64_t v_ld, int gate_kind, void* stream) {
  return lv_masked_attn_mfma(q, k_cache, v_cache, kp, vp, gate, ld_gate, out, cu_q, ctx_lens, block_tables, bt_stride, B,
                             max_new_tokens, H, G, D, Dv, page, window, 0, 0, P, scale, 0.0f, has_sink, nullptr, nsplit, workspace, T,
                             k_ld, v_ld, gate_kind, nullptr, stream);
}

extern "C" int lv_masked_attn_mfma(const void* q, const void* k_cache, const void* v_cache, const void* kp, const void* vp,
                                   const void* gate, int64_t ld_gate, void* out, const int32_t* cu_q, const int32_t* ctx_lens,
                                   const int32_t* block_tables, int bt_stride, int B, int max_new_tokens, int H, int G, int D,
                                   int Dv, int page, int window, int keep_first, int chunk, int P, float scale, float softcap, int has_sink,
                                   const void* sinks, int nsplit, void* workspace, int64_t T, int64_t k_ld, int64_t v_ld,
                                   int gate_kind, const lv_attn_extras* extras, void* stream) {
  if (B == 0 || max_new_tokens <= 0) return 0;
  if (keep_first < 0 || chunk < 0 || (P > 0 && (keep_first > 0 || chunk > 0)))
    return fail(-1, "lv_masked_attn_mfma: kept first tokens and chunks do not combine with pooled blocks");
  if (!(softcap >= 0.0f)) return fail(-1, "lv_masked_attn_mfma: softcap");
  if (sinks != nullptr) has_sink = 1;
  if (!q || !k_cache || !v_cache || !out || !cu_q || !ctx_lens || !block_tables)
    return fail(-1, "lv_window_pool_attn_mfma: null pointer");
  if (P > 0 && (!kp || !vp)) return fail(-1, "lv_window_pool_attn_mfma: pooled blocks without their cache");
  if (B < 0 || H <= 0 || G <= 0 || H % G != 0 || page <= 0 || window <= 0 || bt_stride <= 0)
    return fail(-1, "lv_window_pool_attn_mfma: bad sizes");
  if (D % 16 != 0 || Dv % 16 != 0 || D <= 0 || Dv <= 0 || D > 32 * kMaxK32 || Dv > 16 * kMaxDvb)
    return fail(-2, "lv_window_pool_attn_mfma: head sizes %d / %d (multiples of 16 up to 256)", D, Dv);
  if (gate_kind != LV_MIX_GATE_PER_HEAD && gate_kind != LV_MIX_GATE_PER_CHANNEL)
    return fail(-1, "lv_window_pool_attn_mfma: gate kind %d", gate_kind);
  const int gate_dv = gate_kind == LV_MIX_GATE_PER_HEAD ? 1 : Dv;
  if (gate != nullptr && ld_gate < static_cast<int64_t>(H) * gate_dv) return fail(-1, "lv_window_pool_attn_mfma: gate stride");
  if (k_ld <= 0) k_ld = static_cast<int64_t>(G) * D;
  if (v_ld <= 0) v_ld = static_cast<int64_t>(G) * Dv;
  if (k_ld < static_cast<int64_t>(G) * D || v_ld < static_cast<int64_t>(G) * Dv || k_ld % 8 != 0 || v_ld % 8 != 0 ||
      (reinterpret_cast<uintptr_t>(k_cache) & 15) != 0 || (reinterpret_cast<uintptr_t>(v_cache) & 15) != 0)
    return fail(-1, "lv_window_pool_attn_mfma: row strides or alignment of the caches");
  const bool extended = extras != nullptr && (extras->key_scale != nullptr || extras->dist_bias != nullptr);
  if (extended && (P > 0 || softcap > 0.0f || (extras->dist_bias != nullptr && extras->bias_len <= 0)))
    return fail(-1, "lv_masked_attn_mfma: key factors and distance biases combine with neither pooled blocks nor a softcap");
  const int64_t out_ld = extras != nullptr && extras->out_ld > 0 ? extras->out_ld : static_cast<int64_t>(H) * Dv;
  if (out_ld < static_cast<int64_t>(H) * Dv) return fail(-1, "lv_masked_attn_mfma: output stride");
  const float m0 = has_sink ? 0.0f : -1e30f;
  const int rep = H / G;
  const int ngroups = (rep + 3) / 4;
  WindowMfmaParams p{static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(k_cache),
                     static_cast<const uint16_t*>(v_cache), static_cast<const uint16_t*>(kp),
                     static_cast<const uint16_t*>(vp), static_cast<const uint16_t*>(gate), ld_gate, gate_dv,
                     static_cast<uint16_t*>(out), cu_q, ctx_lens, block_tables, bt_stride, H, G, D, Dv, page, window, P,
                     P > 0 ? (page + P - 1) / P : 0, ngroups, scale, has_sink ? 1.0f : 0.0f,
                     magic(page), magic(P > 0 ? P : 1), magic(Dv / 8), nsplit > 1 ? nsplit : 1, static_cast<float*>(workspace),
                     k_ld, v_ld, m0, keep_first, chunk, static_cast<const float*>(sinks), softcap > 0.0f ? scale / softcap : 0.0f,
                     softcap, extended ? static_cast<const float*>(extras->key_scale) : nullptr,
                     extended ? static_cast<const float*>(extras->dist_bias) : nullptr, extended ? extras->bias_len : 0, out_ld};
  if (nsplit > 1 && (max_new_tokens > kTileQ || workspace == nullptr || T <= 0 || nsplit > kWave))
    return fail(-1, "lv_window_pool_attn_mfma: key splits need one query tile per sequence and a workspace");
  hipStream_t st = as_stream(stream);
  if (nsplit <= 1 && prompt_launch(p, softcap > 0.0f ? kCapped : (extended ? kExtended : kPlain), T, B, max_new_tokens, nsplit < 0, st))
    return launched("lv_masked_attn_mfma");
  auto merge = [&]() {
    const int64_t items = T * H;
    auto launch = [&](auto waves) {
      constexpr int W = decltype(waves)::value;
      window_pool_merge_kernel<W><<<dim3(static_cast<unsigned>((items * W + 3) / 4)), dim3(256), 0, st>>>(
          static_cast<const float*>(workspace), static_cast<const uint16_t*>(gate), ld_gate, gate_dv, static_cast<uint16_t*>(out), items, H, Dv,
          nsplit, out_ld, m0, static_cast<const float*>(sinks));
    };
    if (nsplit > 8) launch(std::integral_constant<int, 4>{});
    else launch(std::integral_constant<int, 1>{});
  };
  if (max_new_tokens == 1 && nsplit >= 0 && decode_launch(p, softcap > 0.0f ? kCapped : (extended ? kExtended : kPlain), B, st)) {
    if (nsplit > 1) merge();
    return launched("lv_masked_attn_mfma");
  }
  size_t shm = static_cast<size_t>(kTileK) * v_row(Dv) * sizeof(uint16_t);
  if (extended) shm += sizeof(float) * (kTileK + (p.dist_bias != nullptr && p.bias_len <= kBiasLds ? 4 * static_cast<size_t>(p.bias_len) : 0));
  dim3 grid(nsplit > 1 ? nsplit : (max_new_tokens + kTileQ - 1) / kTileQ, G * ngroups, B), block(256);
  const bool tiny = D <= 64 && Dv <= 64, small = D <= 128 && Dv <= 128;
#define LVMIX_ATT_FORM(AHEAD, FORM)                                                               \
  do {                                                                                            \
    if (tiny) window_pool_mfma_kernel<AHEAD, 2, 4, FORM><<<grid, block, shm, st>>>(p);            \
    else if (small) window_pool_mfma_kernel<AHEAD, 4, 8, FORM><<<grid, block, shm, st>>>(p);      \
    else window_pool_mfma_kernel<AHEAD, kMaxK32, kMaxDvb, FORM><<<grid, block, shm, st>>>(p);     \
  } while (0)
#define LVMIX_ATT(AHEAD)                                     \
  do {                                                       \
    if (softcap > 0.0f) LVMIX_ATT_FORM(AHEAD, kCapped);      \
    else if (extended) LVMIX_ATT_FORM(AHEAD, kExtended);     \
    else LVMIX_ATT_FORM(AHEAD, kPlain);                      \
  } while (0)
  if (max_new_tokens <= kTileQ) LVMIX_ATT(true);
  else LVMIX_ATT(false);
#undef LVMIX_ATT
#undef LVMIX_ATT_FORM
  if (nsplit > 1) merge();
  return launched("lv_window_pool_attn_mfma");
}

extern "C" int lv_latent_prompt_attn(const void* q, const void* cache, const void* uk, const void* uv, const void* inv_freq, const void* gate,
                                     int64_t ld_gate, int gate_kind, void* out, const int32_t* cu_q, const int32_t* ctx_lens,
                                     const int32_t* block_tables, int bt_stride, int B, int max_new_tokens, int H, int Dn, int Dr, int R,
                                     int page, int window, float scale, const void* sinks, void* stream) {
  if (B == 0 || max_new_tokens <= 0) return 0;
  if (!q || !cache || !uk || !uv || !out || !cu_q || !ctx_lens || !block_tables || (Dr > 0 && !inv_freq))
    return fail(-1, "lv_latent_prompt_attn: null pointer");
  if (gate_kind != LV_MIX_GATE_PER_HEAD && gate_kind != LV_MIX_GATE_PER_CHANNEL) return fail(-1, "lv_latent_prompt_attn: gate kind %d", gate_kind);
  const int gate_dv = gate_kind == LV_MIX_GATE_PER_HEAD ? 1 : Dn;
  if (B < 0 || H <= 0 || H % 4 != 0 || page <= 0 || page % kTileK != 0 || window <= 0 || bt_stride <= 0 || !(scale > 0.0f) ||
      (gate != nullptr && ld_gate < static_cast<int64_t>(H) * gate_dv))
    return fail(-1, "lv_latent_prompt_attn: bad sizes");
  if ((Dn != 64 && Dn != 128) || !((R == 192 && Dr == 64) || (R == 256 && Dr == 0)))
    return fail(-2, "lv_latent_prompt_attn: heads of %d + %d on rows of %d", Dn, Dr, R);
  auto off = [](const void* at, uintptr_t a) { return reinterpret_cast<uintptr_t>(at) % a != 0; };
  if (off(q, 16) || off(cache, 16) || off(uk, 16) || off(uv, 16) || off(out, 8) || (gate != nullptr && gate_dv > 1 && (off(gate, 8) || ld_gate % 4 != 0)))
    return fail(-1, "lv_latent_prompt_attn: alignment");
  const int64_t row = R + Dr;
  LatentParams p{{static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(cache), static_cast<const uint16_t*>(cache), nullptr, nullptr,
                  static_cast<const uint16_t*>(gate), ld_gate, gate_dv, static_cast<uint16_t*>(out), cu_q, ctx_lens, block_tables, bt_stride, H, 1,
                  static_cast<int>(row), R, page, window, 0, 0, H / 4, scale, sinks != nullptr ? 1.0f : 0.0f, magic(page), magic(1), magic(R / 8), 1,
                  nullptr, row, row, -1e30f, 0, 0, static_cast<const float*>(sinks), 0.0f, 0.0f, nullptr, nullptr, 0,
                  static_cast<int64_t>(H) * Dn},
                 static_cast<const uint16_t*>(uk), static_cast<const uint16_t*>(uv), static_cast<const float*>(inv_freq)};
  const int tiles = (max_new_tokens + kPromptQ - 1) / kPromptQ, by = B * (H / 4);
  if (static_cast<int64_t>(tiles) * by >= (1ll << 31)) return fail(-2, "lv_latent_prompt_attn: %d sequences of %d tokens", B, max_new_tokens);
  const dim3 grid(static_cast<unsigned>(tiles) * by), block(256);
  hipStream_t s = as_stream(stream);
  if (R == 192 && Dn == 128) prompt_attn_kernel<256, 192, true, kPlain, 128><<<grid, block, 0, s>>>(p, 4, tiles, by);
  else if (R == 192) prompt_attn_kernel<256, 192, true, kPlain, 64><<<grid, block, 0, s>>>(p, 4, tiles, by);
  else if (Dn == 128) prompt_attn_kernel<256, 256, true, kPlain, 128><<<grid, block, 0, s>>>(p, 4, tiles, by);
  else prompt_attn_kernel<256, 256, true, kPlain, 64><<<grid, block, 0, s>>>(p, 4, tiles, by);
  return launched("lv_latent_prompt_attn");
}
