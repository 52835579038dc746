// Products of up to four rows with a weight, C[M, N] = f(X)[M, K] . W[N, K]^T (+ bias),
// bf16, where f is the RMS norm of X + residual or nothing: the decode step of one or
// a few requests, which is a row of short launches.
//
// Every workgroup makes the normed rows for itself, while its first rows of W are under
// way: for few rows that costs less than a launch. W goes from memory straight to
// registers, where the matrix instruction wants it: 16 rows of 64 bytes a load.
//
// What bounds it: one memory round trip and the launch, then the stream of W. Norm and
// product of one row, us (norm_linear / fused_add_rmsnorm and a product of
// skinny_gemm.hip, W from memory): 1152 x 896 3.1 / 5.5, 9728 x 896 gated 5.8 / 9.0,
// 17920 x 1536 gated 13.2 / 15.8, 6144 x 4096 13.5 / 14.4, 28672 x 4096 gated 42.2 / 42.5;
// of four rows the first three 5.2 / 5.6, 8.7 / 9.4, 13.5 / 15.6, of two rows the others
// 14.0 / 14.5, 43.1 / 42.3.
#include <type_traits>

#include "common.h"

#define NL_ROWS 4  // rows of X at most

namespace {

typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

// s_barrier behind this wave's LDS accesses; loads from memory stay in flight
DEVINL void meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <typename F>
DEVINL void for_rows(int M, F f) {
#pragma unroll
  for (int r = 0; r < NL_ROWS; ++r)
    if (r < M) f(r);
}

DEVINL float silu(float g) { return g / (1.f + __expf(-g)); }

DEVINL float rounded(float v) { return bf16_bits_to_f32(f32_to_bf16_bits(v)); }

}  // namespace

struct NormLinearArgs {
  uint16_t* c;              // [M, N] (gated: [M, N / 2])
  uint16_t* sum;            // [M, K] x + res, or null
  const uint16_t* x;        // [M, K] rows at x_stride
  const uint16_t* res;      // [M, K] or null
  const uint16_t* norm;     // [K] or null: no norm
  const uint16_t* w;        // [N, K]
  const uint16_t* bias;     // [N] or null
  int64_t x_stride, res_stride;
  int M, N, K, tiles;
  float eps;
  bool gated;
};

// The K-steps of 32 are dealt to the waves, S neighbouring ones each; a wave's part of X
// stays in registers, and all of its part of a tile of 16 rows of W is asked for at
// once, that of the next tile as soon as this one's is used. FULL: the steps fill the
// waves. Else those past the end are the last one again with zeros for both operands, as
// W may hold infinities; W's by a mask, which costs 0.5% where a branch around the
// product kept the loads from running ahead (one row of 9000 x 1056 gated 7.05 us and
// 8.3).
template <int WAVES, int S, bool NORM, bool FULL>
__global__ __launch_bounds__(WAVES * 64, 4) void norm_linear_kernel(
    const NormLinearArgs p) {
  __shared__ __attribute__((aligned(16))) float part[2][WAVES][16][16];  // [x row][W row]
  __shared__ float ssq[WAVES][NL_ROWS];
  extern __shared__ __attribute__((aligned(16))) uint16_t xs[];  // [M][K + 32] (NORM)
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l4 = lane >> 4;
  const int steps = p.K / 32;
  const int m = min(l15, p.M - 1);  // a lane's row of X
  uint32_t off[S];
#pragma unroll
  for (int s = 0; s < S; ++s)
    off[s] = min(wid * S + s, steps - 1) * 32 + l4 * 8;

  // a thread has at most 8 neighbouring values of each row: K <= 8 * 64 * WAVES
  bf16x8 xv[NORM ? NL_ROWS : 1], rv[NORM ? NL_ROWS : 1], gain;
  bf16x8v xf[S], wf[S];
  const int k0 = tid * 8;
  if constexpr (NORM) {
    if (k0 < p.K) {
      for_rows(p.M, [&](int r) {
        xv[r] = load_bf16x8(p.x + r * p.x_stride + k0);
        if (p.res != nullptr) rv[r] = load_bf16x8(p.res + r * p.res_stride + k0);
      });
      gain = load_bf16x8(p.norm + k0);
    }
  } else {
#pragma unroll
    for (int s = 0; s < S; ++s)
      xf[s] = *reinterpret_cast<const bf16x8v*>(p.x + m * p.x_stride + off[s]);
  }
  const int side = p.gated ? 8 : 16, N1 = p.gated ? p.N / 2 : p.N;
  auto row = [&](int tile) {
    const int n = min(tile * side + (l15 & (side - 1)), N1 - 1);
    return p.w + (size_t)(l15 < side ? n : n + N1) * p.K;
  };
  auto load_w = [&](const uint16_t* r, int s) {
    wf[s] = *reinterpret_cast<const bf16x8v*>(r + off[s]);
  };
  {
    const uint16_t* r = row(blockIdx.x);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      load_w(r, s);
      asm volatile("" ::: "memory");  // asked for in the order of their use
    }
  }
  if constexpr (NORM) {
    for_rows(p.M, [&](int r) {
      float v[8], ss = 0.f;
      if (k0 < p.K) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = bf16x8_get(xv[r], j);
        if (p.res != nullptr) {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] += bf16x8_get(rv[r], j);
          store_bf16x8(&xv[r], v);
          if (blockIdx.x == 0)
            *reinterpret_cast<int4*>(p.sum + (size_t)r * p.K + k0) = xv[r].raw;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) ss = fmaf(v[j], v[j], ss);
      }
      ss = wave_reduce_sum(ss);
      if (lane == 0) ssq[wid][r] = ss;
    });
    meet();
    if (k0 < p.K)
      for_rows(p.M, [&](int r) {
        float all = 0.f;
#pragma unroll
        for (int v = 0; v < WAVES; ++v) all += ssq[v][r];
        const float rstd = rsqrtf(all / p.K + p.eps);
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          v[j] = bf16x8_get(xv[r], j) * rstd * bf16x8_get(gain, j);
        store_bf16x8(xs + r * (p.K + 32) + k0, v);
      });
    meet();
#pragma unroll
    for (int s = 0; s < S; ++s)
      xf[s] = *reinterpret_cast<const bf16x8v*>(xs + m * (p.K + 32) + off[s]);
  }
  if (!FULL)
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (wid * S + s >= steps) xf[s] = 0;

  int buf = 0;
  for (int tile = blockIdx.x; tile < p.tiles; tile += gridDim.x) {
    const bool more = tile + gridDim.x < (unsigned)p.tiles;
    const uint16_t* r = row(tile + gridDim.x);
    f32x4v acc = {};
#pragma unroll
    for (int s = 0; s < S; ++s) {
      u32x4v w = __builtin_bit_cast(u32x4v, wf[s]);
      if (!FULL) w &= wid * S + s < steps ? ~0u : 0u;
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v, w),
                                                    xf[s], acc, 0, 0, 0);
      if (more) load_w(r, s);
    }
    *reinterpret_cast<f32x4v*>(&part[buf][wid][l15][l4 * 4]) = acc;
    meet();
    // four lanes a result, each the sums of a quarter of the waves
    for (int e = tid; e < p.M * side * 4; e += WAVES * 64) {
      const int q = e & 3, n = (e >> 2) % side, row = (e >> 2) / side;
      auto sum = [&](int n) {
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < WAVES / 4; ++k) v += part[buf][q * (WAVES / 4) + k][row][n];
        v += __shfl_xor(v, 1, WAVE_SIZE);
        return v + __shfl_xor(v, 2, WAVE_SIZE);
      };
      float v = sum(n), u = p.gated ? sum(n + 8) : 0.f;
      const int at = tile * side + n;
      if (q == 0 && at < N1) {
        if (p.bias != nullptr) {
          v += bf16_bits_to_f32(p.bias[at]);
          if (p.gated) u += bf16_bits_to_f32(p.bias[N1 + at]);
        }
        p.c[(size_t)row * N1 + at] =
            f32_to_bf16_bits(p.gated ? silu(rounded(v)) * rounded(u) : v);
      }
    }
    buf ^= 1;
  }
}

// Where it is the faster side, see above. With the norm: any rows of up to 2048, where
// four or eight waves hold X; two rows of up to 4096, whose 16 waves leave one
// workgroup a CU (four rows of 5120 x 3072 13.1 / 13.0, 4608 x 3584 14.8 / 13.9), and
// then not the longest streams (one row of 37888 x 3584 gated 60 / 58). The product
// alone: short rows (one row of 896 x 896 3.2 / 3.4, 2048 x 1536 4.2 / 4.8, 17920 x
// 1536 gated 14.9 / 16.2; but 16384 x 2048 gated 16.5 / 15.3, 3584 x 2560 6.8 / 6.3).
extern "C" bool norm_linear_takes(int64_t M, int64_t N, int64_t K, bool norm) {
  if (M < 1 || M > NL_ROWS || N < 1 || K < 32 || K % 32) return false;
  if (!norm) return K <= 1536 && N <= 20000;
  return N <= 1 << 20 && (K <= 2048 || (K <= 4096 && M <= 2 && N * K <= 120000000));
}

extern "C" void launch_norm_linear(
    void* c, void* sum, const void* x, const void* res, const void* norm,
    const void* w, const void* bias, float eps, int M, int N, int K,
    int64_t x_stride, int64_t res_stride, bool gated, hipStream_t stream) {
  const int steps = K / 32;
  NormLinearArgs p{(uint16_t*)c, (uint16_t*)sum, (const uint16_t*)x,
                   (const uint16_t*)res, (const uint16_t*)norm, (const uint16_t*)w,
                   (const uint16_t*)bias, x_stride, res_stride, M, N, K,
                   gated ? ceil_div(N / 2, 8) : ceil_div(N, 16), eps, gated};
  auto run = [&](auto wv, auto sv) {
    constexpr int W = decltype(wv)::value, S = decltype(sv)::value;
    const int slots = 4096 / W;  // workgroups that the chip holds: 4 waves a SIMD
    const int grid = min(p.tiles, slots);
    auto go = [&](auto full) {
      constexpr bool F = decltype(full)::value;
      if (norm == nullptr) {
        if constexpr (W * S <= 48)
          norm_linear_kernel<W, S, false, F><<<grid, W * 64, 0, stream>>>(p);
      } else {
        norm_linear_kernel<W, S, true, F>
            <<<grid, W * 64, (size_t)M * (K + 32) * 2, stream>>>(p);
      }
    };
    if (steps == W * S) go(std::true_type{});
    else go(std::false_type{});
  };
#define PICK(W, S) run(std::integral_constant<int, W>{}, std::integral_constant<int, S>{})
  if (steps <= 16) PICK(4, 4);
  else if (steps <= 28) PICK(4, 7);
  else if (steps <= 32) PICK(4, 8);
  else if (steps <= 48) PICK(8, 6);
  else if (steps <= 64) PICK(8, 8);
  else if (steps <= 96) PICK(16, 6);
  else PICK(16, 8);
#undef PICK
}
