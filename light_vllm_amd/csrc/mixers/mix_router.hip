// Router logits of prompt steps: f32 [T, E] = h w^T for bf16 activations h and f32 weights w, f32 products and sums on
// v_mfma_f32_16x16x4_f32, without a widened copy of the activations.
//
// Tokens whose experts nearly tie take one or the other by the order of these sums, so the order is that of the f32 product this stands in
// for: one chain over k in blocks of 16, product i of a block on its entries i, 4 + i, 8 + i and 12 + i. The same bits at widths of 512, 1024, 2048 and 4096
// for 32 experts and 4500 (4096: 6000) to 32768 tokens, 64 experts and 9000 to 16384; beyond 16384 tokens the product of 64 experts sums otherwise.
//
// Bound by the chain of f32 products (16 x 16 x 4: 32 clocks on a SIMD; 14 us at 16384 x 2048 x 32) and by reading h once (67 MB there, 12 us).
// A workgroup of eight waves takes 64 rows: four waves' worth of 16 rows, by halves of the experts, so that a SIMD has two chains to
// turn to. Steps of 64 k pass through LDS, four are on their way in registers, and a step's
// fragments are read during the one before it. 16384 x 2048 x 32 in a layer: widening and product 67 us -> 33; with a step's fragments read in front
// of its products 29 for 26 by itself.
#include "mix_common.h"

namespace lvmix {

typedef float router_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t router_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t router_u32x4 __attribute__((ext_vector_type(4)));
constexpr int kRouterRows = 64, kRouterAhead = 4;

struct RouterParams {
  const uint16_t* h;
  const float* w;
  float* out;
  int64_t ldh;
  int T, W, E;
};

// NC: blocks of 16 experts of a wave; the second half of the waves takes the blocks behind those of the first.
template <int NC>
__global__ __launch_bounds__(512, 2) void router_tile_kernel(RouterParams p) {
  constexpr int XB = kRouterRows * 128, WB = 32 * NC * 256;          // bytes of a step: rows of 64 bf16, rows of 64 f32
  __shared__ __attribute__((aligned(16))) uint8_t slots[kRouterAhead][XB + WB];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, quad = lane >> 4;
  const int row0 = static_cast<int>(blockIdx.x) * kRouterRows, rg = w & 3, cg = w >> 2;
  const int steps = p.W / 64;
  // Loads: a wave brings 8 rows of h and NC times 4 rows of w a step. The 16-byte piece c of row i of h sits at c ^ ((i >> 1) & 7), of w at
  // c ^ (i & 15): reads of 16 rows meet all banks.
  const int hrow = 8 * w + (lane >> 3), hpiece = (lane & 7) ^ ((hrow >> 1) & 7);
  const uint16_t* const hfrom = p.h + static_cast<int64_t>(min(row0 + hrow, p.T - 1)) * p.ldh + 8 * hpiece;     // rows past the end: the last one, not stored
  const float* wfrom[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int e = 4 * (w + 8 * i) + (lane >> 4);
    wfrom[i] = p.w + static_cast<int64_t>(min(e, p.E - 1)) * p.W + 4 * ((lane & 15) ^ (e & 15));
  }
  router_u32x4 hreg[kRouterAhead];
  router_f32x4 wreg[kRouterAhead][NC];
  auto request = [&](auto place, int s) __attribute__((always_inline)) {
    constexpr int k = decltype(place)::value;
    const int at = min(s, steps - 1);                                // past the end: some step, never used
    hreg[k] = *reinterpret_cast<const router_u32x4*>(hfrom + 64 * at);
#pragma unroll
    for (int i = 0; i < NC; ++i) wreg[k][i] = *reinterpret_cast<const router_f32x4*>(wfrom[i] + 64 * at);
  };
  auto stage = [&](auto place, int slot) __attribute__((always_inline)) {
    constexpr int k = decltype(place)::value;
    *reinterpret_cast<router_u32x4*>(slots[slot] + 1024 * w + 16 * lane) = hreg[k];
#pragma unroll
    for (int i = 0; i < NC; ++i) *reinterpret_cast<router_f32x4*>(slots[slot] + XB + 1024 * (w + 8 * i) + 16 * lane) = wreg[k][i];
  };
  router_f32x4 acc[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) acc[j] = router_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int x_off = (16 * rg + r) * 128, y_off = XB + (16 * NC * cg + r) * 256;
  struct Frags { router_u32x2 x[4]; router_f32x4 y[4][NC]; };
  auto fetch = [&](int slot, Frags& f) __attribute__((always_inline)) {
    const uint8_t* const at = slots[slot];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      f.x[b] = *reinterpret_cast<const router_u32x2*>(at + x_off + (((2 * b + (quad >> 1)) ^ ((r >> 1) & 7)) * 16) + 8 * (quad & 1));
#pragma unroll
      for (int j = 0; j < NC; ++j) f.y[b][j] = *reinterpret_cast<const router_f32x4*>(at + y_off + 16 * 256 * j + (((4 * b + quad) ^ r) * 16));
    }
  };
  auto products = [&](const Frags& f, int from) __attribute__((always_inline)) {
#pragma unroll
    for (int b = from; b < from + 2; ++b) {
      const float v[4] = {__builtin_bit_cast(float, f.x[b].x << 16), __builtin_bit_cast(float, f.x[b].x & 0xffff0000u),
                          __builtin_bit_cast(float, f.x[b].y << 16), __builtin_bit_cast(float, f.x[b].y & 0xffff0000u)};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NC; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.y[b][j][i], v[i], acc[j], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // Step s (s % 4 = K): its fragments are in registers. Those of step s + 1 are read, step s + 2 goes from registers to its slot, which
  // everyone read during step s - 3, in front of a barrier, and step s + 6 is asked for in its place.
  Frags f0, f1;
  auto step = [&](auto K, const Frags& f, Frags& next, int s) __attribute__((always_inline)) {
    constexpr int k = decltype(K)::value;
    fetch((k + 1) % 4, next);
    __builtin_amdgcn_sched_barrier(0);
    products(f, 0);
    stage(std::integral_constant<int, (k + 2) % 4>{}, (k + 2) % 4);
    request(std::integral_constant<int, (k + 2) % 4>{}, s + 2 + kRouterAhead);
    __builtin_amdgcn_sched_barrier(0);
    products(f, 2);
    __syncthreads();
  };
  using K0 = std::integral_constant<int, 0>;
  using K1 = std::integral_constant<int, 1>;
  using K2 = std::integral_constant<int, 2>;
  using K3 = std::integral_constant<int, 3>;
  auto ask = [&](auto k, int s) __attribute__((always_inline)) {     // (the loop counts on their order)
    request(k, s);
    __builtin_amdgcn_sched_barrier(0);
  };
  ask(K0{}, 0);
  ask(K1{}, 1);
  ask(K2{}, 2);
  ask(K3{}, 3);
  stage(K0{}, 0);
  ask(K0{}, 4);
  stage(K1{}, 1);
  ask(K1{}, 5);
  __syncthreads();
  fetch(0, f0);
  for (int s = 0; s < steps; s += 4) {                               // (W is a multiple of 256)
    step(K0{}, f0, f1, s);
    step(K1{}, f1, f0, s + 1);
    step(K2{}, f0, f1, s + 2);
    step(K3{}, f1, f0, s + 3);
  }
  const int row = row0 + 16 * rg + r;
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int e = 16 * (NC * cg + j) + 4 * quad;                     // E is a multiple of 16
    if (row < p.T && e < p.E) *reinterpret_cast<router_f32x4*>(p.out + static_cast<int64_t>(row) * p.E + e) = acc[j];
  }
}

}  // namespace lvmix

using namespace lvmix;

extern "C" int lv_router_tiles(const void* h, int64_t ld_h, const void* router_w, void* logits, int64_t T, int W, int E, void* stream) {
  if (T == 0) return 0;
  if (!h || !router_w || !logits || T < 0 || T >= (int64_t{1} << 30) || W <= 0 || W % 256 != 0 || E < 16 || E > 64 || E % 16 != 0 || ld_h < W ||
      ld_h % 8 != 0 || ((reinterpret_cast<uintptr_t>(h) | reinterpret_cast<uintptr_t>(router_w) | reinterpret_cast<uintptr_t>(logits)) & 15) != 0)
    return fail(-1, "lv_router_tiles: %d experts, width %d, row stride %lld or alignment", E, W, static_cast<long long>(ld_h));
  const RouterParams p{static_cast<const uint16_t*>(h), static_cast<const float*>(router_w), static_cast<float*>(logits), ld_h,
                       static_cast<int>(T), W, E};
  const dim3 grid(static_cast<unsigned>((T + kRouterRows - 1) / kRouterRows)), block(512);
  if (E <= 32) router_tile_kernel<1><<<grid, block, 0, as_stream(stream)>>>(p);
  else router_tile_kernel<2><<<grid, block, 0, as_stream(stream)>>>(p);
  return launched("lv_router_tiles");
}
