// Products of few rows with a large weight: C[M, N] = X[M, K] . W[N, K]^T (+ bias),
// bf16 or (scaled per tensor) fp8.
//
// A decode step's projections: the weight's stream is the bound. A workgroup
// takes NT rows of W; its waves deal the 128-byte columns of those rows among
// them (wave w the columns w, w + WAVES, ..), so that it reads long runs of
// each row, and every wave is on its own: W and X go global -> LDS directly
// into its own ring of STAGES, and it waits for its own copies only. No barrier
// until the sums of the waves are added at the end. A head start of its own
// rotates every workgroup's columns: rows lie a power of two apart, and all
// workgroups at one column would wait for the same L2 channels (28672 x 4096, 8
// rows: 44 to 40 us).
//
// What bounds it: up to 8 rows the stream from memory (28672 x 4096 in 39 us, 6.0
// TB/s; 4096 x 14336 in 22 us; the library 52 and 25), for small weights one round
// trip and the launch (896 x 896 in 3.3 us, before 5.5); with more rows what L2
// delivers, W and X together 8.8 TB/s.

#include <type_traits>

#include "common.h"

typedef float f32x16v __attribute__((ext_vector_type(16)));
typedef short s16x4v __attribute__((ext_vector_type(4)));
typedef int i32x4n __attribute__((ext_vector_type(4)));
typedef int i32x8n __attribute__((ext_vector_type(8)));

namespace {

DEVINL void copy16_to_lds(const void* src, void* dst) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)src,
      (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// 32 fp8 values of an operand; their order in K is that of the other operand's
DEVINL i32x8n join(bf16x8v lo, bf16x8v hi) {
  return __builtin_shufflevector(__builtin_bit_cast(i32x4n, lo),
                                 __builtin_bit_cast(i32x4n, hi), 0, 1, 2, 3, 4, 5,
                                 6, 7);
}

template <int N>
DEVINL void wait_copies() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N & 48) << 10));
  asm volatile("" ::: "memory");
}

// Two to six operands of 16 bytes a lane, at at + 2048 t and x_at + 2048 u. Not
// plain loads: before those the compiler waits for every copy in flight.
template <int A, int B>
DEVINL void read_operands(const uint32_t at, const uint32_t x_at, bf16x8v (&a)[A],
                          bf16x8v (&b)[B]) {
  static_assert((A == 1 || A == 2 || A == 4) && (B == 1 || B == 2 || B == 4), "");
  if constexpr (A == 4) {
    asm volatile(
        "ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:2048\n\t"
        "ds_read_b128 %2, %4 offset:4096\n\tds_read_b128 %3, %4 offset:6144\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3])
        : "v"(at) : "memory");
  }
  if constexpr (B == 4) {
    asm volatile(
        "ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:2048\n\t"
        "ds_read_b128 %2, %4 offset:4096\n\tds_read_b128 %3, %4 offset:6144\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2]), "=&v"(b[3])
        : "v"(x_at) : "memory");
  }
  if constexpr (A == 1 && B == 1)
    asm volatile(
        "ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(a[0]), "=&v"(b[0]) : "v"(at), "v"(x_at) : "memory");
  if constexpr (A == 2 && B == 1)
    asm volatile(
        "ds_read_b128 %0, %3\n\tds_read_b128 %1, %3 offset:2048\n\t"
        "ds_read_b128 %2, %4\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(a[0]), "=&v"(a[1]), "=&v"(b[0])
        : "v"(at), "v"(x_at) : "memory");
  if constexpr (A == 1 && B == 2)
    asm volatile(
        "ds_read_b128 %0, %3\n\tds_read_b128 %1, %4\n\t"
        "ds_read_b128 %2, %4 offset:2048\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(a[0]), "=&v"(b[0]), "=&v"(b[1])
        : "v"(at), "v"(x_at) : "memory");
  if constexpr (A == 2 && B == 2)
    asm volatile(
        "ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:2048\n\t"
        "ds_read_b128 %2, %5\n\tds_read_b128 %3, %5 offset:2048\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0]), "=&v"(a[1]), "=&v"(b[0]), "=&v"(b[1])
        : "v"(at), "v"(x_at) : "memory");
  if constexpr (A == 2 && B == 4)
    asm volatile(
        "ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:2048\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0]), "=&v"(a[1]) : "v"(at) : "memory");
  if constexpr (A == 4 && B == 2)
    asm volatile(
        "ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:2048\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(b[0]), "=&v"(b[1]) : "v"(x_at) : "memory");
  if constexpr (A == 1 && B == 4)
    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(a[0]) : "v"(at) : "memory");
  if constexpr (A == 4 && B == 1)
    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(b[0]) : "v"(x_at) : "memory");
}

}  // namespace

// Gated: W is [gate rows | up rows], N of both together; tiles take as many of
// each, and the result is silu(gate) * up of the rounded products, [M, N / 2].
DEVINL uint16_t silu_mul(float g, float u) {
  g = bf16_bits_to_f32(f32_to_bf16_bits(g));
  u = bf16_bits_to_f32(f32_to_bf16_bits(u));
  return f32_to_bf16_bits(g / (1.f + __expf(-g)) * u);
}

DEVINL float biased(float v, const uint16_t* bias, int n) {
  return bias != nullptr ? v + bf16_bits_to_f32(bias[n]) : v;
}

// XR: rows of X staged, a multiple of 8 that holds M.
template <bool FP8, int NT, int XR, int WAVES, int STAGES>
__global__ __launch_bounds__(WAVES * 64) void skinny_gemm_kernel(
    uint16_t* __restrict__ c,          // [M, N] bf16 rows at c_stride
    const uint8_t* __restrict__ x,     // [M, K] rows at x_stride bytes
    const uint8_t* __restrict__ w,     // [N, K]
    const uint16_t* __restrict__ bias, // [N] or null
    const float* __restrict__ x_scale, const float* __restrict__ w_scale,
    const int M_all, const int N, const int row_bytes, const int64_t x_stride,
    const int64_t c_stride, const int64_t x_batch, const int64_t c_batch,
    const bool gated) {
  constexpr int ROWS = NT + XR;
  constexpr int NI = ROWS / 8;  // copies a stage: 8 rows of 128 bytes each
  constexpr int MT = (XR + 15) / 16;
  constexpr int MP = MT * 16;
  constexpr int AT = (NT + 15) / 16;  // NT 8: the operand's upper rows are the lower
  constexpr int RING = ROWS * 128;  // a wave's stage
  __shared__ __attribute__((aligned(128))) uint8_t S[WAVES * STAGES * RING];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l4 = lane >> 4;
  // rows of W that lie together in a tile, and in W
  const int side = gated ? NT / 2 : NT, N1 = gated ? N / 2 : N;
  const int n0 = blockIdx.x * side;
  const int M = min(XR, M_all - (int)blockIdx.z * XR);
  x += blockIdx.y * x_batch + blockIdx.z * XR * x_stride;
  c += blockIdx.y * c_batch + blockIdx.z * XR * c_stride;
  const uint8_t* wb = w + ((size_t)blockIdx.y * N + n0) * row_bytes;

  // chunk (row, j) of a stage lies at j ^ (row / 2 & 7) in the row's 128 bytes
  uint32_t at[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = i * 8 + (lane >> 3);
    const int j = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    const int up = r < side ? 0 : N1 - side;  // from a gate's row to an up row
    at[i] = r < NT ? (uint32_t)(min(r, N1 - 1 - n0 + (r < side ? 0 : side)) + up) *
                             row_bytes + j
                   : (uint32_t)min(r - NT, M - 1) * (uint32_t)x_stride + j;
  }
  const int cols = row_bytes / 128;
  const int mine = (cols - wid + WAVES - 1) / WAVES;

  const int rot0 = mine > 0 ? (int)((blockIdx.x >> 3) * 3 % mine) : 0;
  uint8_t* ring = S + wid * (STAGES * RING);
  auto issue = [&](int i, int place) __attribute__((always_inline)) {
    int t = min(i, mine - 1) + rot0;
    if (t >= mine) t -= mine;
    const int k = (t * WAVES + wid) * 128;
    uint8_t* dst = ring + place * RING;
#pragma unroll
    for (int q = 0; q < NI; ++q)
      copy16_to_lds((q * 8 < NT ? wb : x) + k + at[q], dst + q * 1024);
  };

  f32x4v acc[AT][MT] = {};
  const uint32_t ring_at =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)ring;
  const int wr = l15 & (NT < 16 ? NT - 1 : 15);
  const int xr = l15 & (XR < 16 ? XR - 1 : 15);
  const uint32_t a_at = ring_at + wr * 128 + (l4 ^ ((wr >> 1) & 7)) * 16;
  const uint32_t b_at =
      ring_at + (NT + xr) * 128 + (l4 ^ (((NT + xr) >> 1) & 7)) * 16;
  int place = 0, next = STAGES - 1;
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i)
    if (mine > 0) issue(i, i);
  for (int i = 0; i < mine; ++i) {
    wait_copies<(STAGES - 2) * NI>();
    // into the place read in the turn before: its operands are in registers
    issue(i + STAGES - 1, next);
    bf16x8v a[2][AT], b[2][MT];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      read_operands((a_at + place * RING) ^ (ks * 64),
                    (b_at + place * RING) ^ (ks * 64), a[ks], b[ks]);
#pragma unroll
    for (int t = 0; t < AT; ++t)
#pragma unroll
      for (int u = 0; u < MT; ++u) {
        if constexpr (FP8) {
          acc[t][u] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
              join(a[0][t], a[1][t]), join(b[0][u], b[1][u]), acc[t][u], 0, 0, 0,
              0x7f7f7f7f, 0, 0x7f7f7f7f);
        } else {
#pragma unroll
          for (int ks = 0; ks < 2; ++ks)
            acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                a[ks][t], b[ks][u], acc[t][u], 0, 0, 0);
        }
      }
    place = place + 1 == STAGES ? 0 : place + 1;
    next = next + 1 == STAGES ? 0 : next + 1;
  }
  wait_copies<0>();
  __syncthreads();
  float* part = reinterpret_cast<float*>(S);
  static_assert(MP * NT * 4 <= STAGES * RING, "");
#pragma unroll
  for (int t = 0; t < AT; ++t)
#pragma unroll
    for (int u = 0; u < MT; ++u)
      if (NT >= 16 || l4 * 4 < NT)
        *reinterpret_cast<f32x4v*>(
            part + ((wid * MP + u * 16 + l15) * NT + t * 16 + l4 * 4)) = acc[t][u];
  __syncthreads();
  const float scale = FP8 ? x_scale[0] * w_scale[0] : 1.f;
  const int quads = side / 4;
  for (int e = tid; e < M * quads; e += WAVES * 64) {
    const int m = e / quads, n = e % quads * 4;
    if (n0 + n >= N1) continue;
    auto sum = [&](int n) {
      f32x4v s = {};
#pragma unroll
      for (int v = 0; v < WAVES; ++v)
        s += *reinterpret_cast<const f32x4v*>(part + ((v * MP + m) * NT + n));
      return FP8 ? s * scale : s;
    };
    const f32x4v s = sum(n), u = gated ? sum(n + side) : s;
    uint16_t o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float f = biased(s[r], bias, n0 + n + r);
      o[r] = gated ? silu_mul(f, biased(u[r], bias, N1 + n0 + n + r))
                   : f32_to_bf16_bits(f);
    }
    *reinterpret_cast<uint2*>(c + (size_t)m * c_stride + n0 + n) =
        make_uint2(o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16);
  }
}

// ---- to 128 rows -------------------------------------------------------------------------
// X is as large as W's part: the waves of a workgroup share its tile and take 32
// rows of W each; one barrier a stage. Where W has few rows, K is split over
// workgroups, whose fp32 parts a second kernel adds up. W's stream bounds it, 28672
// x 4096 at 96 rows in 47 us or 5.0 TB/s, and for small weights the second launch.

// Stage operands: 16 bytes of the wave's 32 rows of W, and of 32 XT rows of X
template <int XT>
DEVINL void read_stage(bf16x8v& a, bf16x8v (&b)[XT], uint32_t at, uint32_t x_at) {
  static_assert(XT >= 1 && XT <= 4, "");
  if constexpr (XT == 1)
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(a), "=&v"(b[0]) : "v"(at), "v"(x_at) : "memory");
  if constexpr (XT == 2)
    asm volatile("ds_read_b128 %0, %3\n\tds_read_b128 %1, %4\n\t"
                 "ds_read_b128 %2, %4 offset:4096\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(a), "=&v"(b[0]), "=&v"(b[1])
                 : "v"(at), "v"(x_at) : "memory");
  if constexpr (XT == 3)
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\t"
                 "ds_read_b128 %2, %5 offset:4096\n\t"
                 "ds_read_b128 %3, %5 offset:8192\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(a), "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2])
                 : "v"(at), "v"(x_at) : "memory");
  if constexpr (XT == 4)
    asm volatile("ds_read_b128 %0, %5\n\tds_read_b128 %1, %6\n\t"
                 "ds_read_b128 %2, %6 offset:4096\n\t"
                 "ds_read_b128 %3, %6 offset:8192\n\t"
                 "ds_read_b128 %4, %6 offset:12288\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(a), "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2]), "=&v"(b[3])
                 : "v"(at), "v"(x_at) : "memory");
}

template <bool FP8, int XT, int W, int STAGES>
__global__ __launch_bounds__(W * 64) void skinny_split_kernel(
    uint16_t* __restrict__ c, float* __restrict__ part,  // [splits, M, N] or null
    const uint8_t* __restrict__ x, const uint8_t* __restrict__ w,
    const uint16_t* __restrict__ bias, const float* __restrict__ x_scale,
    const float* __restrict__ w_scale, const int M, const int N,
    const int row_bytes, const int64_t x_stride, const int64_t c_stride,
    const bool gated) {
  constexpr int NT = W * 32;
  constexpr int ROWS = NT + XT * 32;
  // copies a wave and stage: its rows of W, some of X
  constexpr int NX = (XT * 4 + W - 1) / W;
  constexpr int NI = 4 + NX;
  constexpr int RING = ROWS * 128;
  __shared__ __attribute__((aligned(128))) uint8_t S[STAGES * RING];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, l31 = lane & 31;
  // gated: a wave takes 16 rows of gate and 16 of up, which land in one lane
  const int side = gated ? 16 : 32, N1 = gated ? N / 2 : N;
  const int n0 = blockIdx.x * (W * side);

  // this workgroup's columns of 128 bytes
  const int cols = row_bytes / 128;
  const int c0 = (int)((int64_t)cols * blockIdx.y / gridDim.y);
  const int mine = (int)((int64_t)cols * (blockIdx.y + 1) / gridDim.y) - c0;
  const uint8_t* wb = w + (size_t)n0 * row_bytes + (size_t)c0 * 128;
  const uint8_t* xb = x + (size_t)c0 * 128;
  uint32_t at[NI];
  // eight rows of X: where the waves do not divide them, the last are copied twice
  auto x_rows = [&](int i) { return min(wid + W * i, XT * 4 - 1) * 8; };
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = (i < 4 ? i * 8 : x_rows(i - 4)) + (lane >> 3);
    const int j = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    const int n = min(wid * side + r % side, N1 - 1 - n0) + r / side * N1;
    at[i] = i < 4 ? (uint32_t)n * row_bytes + j
                  : (uint32_t)min(r, M - 1) * (uint32_t)x_stride + j;
  }
  // one head start a workgroup, see skinny_gemm_kernel
  const int rot = (int)((blockIdx.x >> 3) * 3 % mine);
  auto issue = [&](int i, int place) __attribute__((always_inline)) {
    int t = min(i, mine - 1) + rot;
    if (t >= mine) t -= mine;
    uint8_t* dst = S + place * RING;
#pragma unroll
    for (int q = 0; q < NI; ++q)
      copy16_to_lds((q < 4 ? wb : xb) + t * 128 + at[q],
                    dst + (q < 4 ? wid * 32 + q * 8 : NT + x_rows(q - 4)) * 128);
  };
  f32x16v acc[XT] = {};
  const uint32_t base =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)S;
  const uint32_t j0 = (half ^ ((l31 >> 1) & 7)) * 16;
  const uint32_t a_at = base + (wid * 32 + l31) * 128 + j0;
  const uint32_t b_at = base + (NT + l31) * 128 + j0;
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i) issue(i, i);
  int place = 0, next = STAGES - 1;
  for (int i = 0; i < mine; ++i) {
    wait_copies<(STAGES - 2) * NI>();
    // every wave's copies have landed, and every wave is done with the place
    // that is filled next: its operands are in registers
    __builtin_amdgcn_s_barrier();
    issue(i + STAGES - 1, next);
#pragma unroll
    for (int ks = 0; ks < 4; ks += 2) {
      bf16x8v a[2], b[2][XT];
#pragma unroll
      for (int k = 0; k < 2; ++k)
        read_stage<XT>(a[k], b[k], (a_at + place * RING) ^ ((ks + k) * 32),
                       (b_at + place * RING) ^ ((ks + k) * 32));
#pragma unroll
      for (int t = 0; t < XT; ++t) {
        if constexpr (FP8) {
          acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
              join(a[0], a[1]), join(b[0][t], b[1][t]), acc[t], 0, 0, 0,
              0x7f7f7f7f, 0, 0x7f7f7f7f);
        } else {
#pragma unroll
          for (int k = 0; k < 2; ++k)
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[k], b[k][t], acc[t],
                                                             0, 0, 0);
        }
      }
    }
    place = place + 1 == STAGES ? 0 : place + 1;
    next = next + 1 == STAGES ? 0 : next + 1;
  }
  wait_copies<0>();
  const float scale = FP8 ? x_scale[0] * w_scale[0] : 1.f;
#pragma unroll
  for (int t = 0; t < XT; ++t) {
    const int m = t * 32 + l31;
    if (m >= M) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = 8 * q + 4 * half;  // of the wave's 32
      const int n = n0 + wid * side + row % side;
      if (n >= N1) continue;
      f32x4v v, u;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = acc[t][4 * q + r];
        u[r] = acc[t][(4 * q + 8 + r) & 15];
      }
      if (FP8) v *= scale;
      if (part != nullptr) {
        *reinterpret_cast<f32x4v*>(part + ((size_t)blockIdx.y * M + m) * N + n +
                                   row / side * N1) = v;
        continue;
      }
      if (row >= side) continue;
      if (FP8) u *= scale;
      uint16_t o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float f = biased(v[r], bias, n + r);
        o[r] = gated ? silu_mul(f, biased(u[r], bias, N1 + n + r))
                     : f32_to_bf16_bits(f);
      }
      *reinterpret_cast<uint2*>(c + (size_t)m * c_stride + n) =
          make_uint2(o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16);
    }
  }
}

__global__ __launch_bounds__(256) void skinny_sum_kernel(
    uint16_t* __restrict__ c, const float* __restrict__ part,
    const uint16_t* __restrict__ bias, const int splits, const int M, const int N,
    const int64_t c_stride, const bool gated) {
  const int N1 = gated ? N / 2 : N;
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const int64_t all = (int64_t)M * N;
  const int m = (int)(e / N1), n = (int)(e % N1);
  if (m >= M) return;
  auto sum = [&](int n) {
    const float* src = part + (int64_t)m * N + n;
    f32x4v s = {};
#pragma unroll 8
    for (int k = 0; k < splits; ++k)
      s += *reinterpret_cast<const f32x4v*>(src + k * all);
    return s;
  };
  const f32x4v s = sum(n);
  f32x4v u = s;
  if (gated) u = sum(N1 + n);
  uint16_t o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float f = biased(s[r], bias, n + r);
    o[r] = gated ? silu_mul(f, biased(u[r], bias, N1 + n + r)) : f32_to_bf16_bits(f);
  }
  *reinterpret_cast<uint2*>(c + (size_t)m * c_stride + n) =
      make_uint2(o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16);
}

// The sum and what it is added to behind a shard's last layer, rounded before and after
// as the two launches do. The launches bound it: 40 rows of 7168 8.7 us in two, 4.1 in one.
__global__ __launch_bounds__(256) void skinny_add_kernel(
    uint16_t* __restrict__ c, const float* __restrict__ part,
    const uint16_t* __restrict__ residual, const int splits, const int M, const int N,
    const int64_t res_stride) {
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const int64_t all = (int64_t)M * N;
  if (e >= all) return;
  const int m = (int)(e / N), n = (int)(e % N);
  const uint2 r = *reinterpret_cast<const uint2*>(residual + m * res_stride + n);
  f32x4v s = {};
#pragma unroll 8
  for (int k = 0; k < splits; ++k)
    s += *reinterpret_cast<const f32x4v*>(part + k * all + e);
  uint16_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    o[i] = f32_to_bf16_bits(bf16_bits_to_f32(f32_to_bf16_bits(s[i])) +
                            bf16_bits_to_f32((uint16_t)((i < 2 ? r.x : r.y) >> 16 * (i & 1))));
  *reinterpret_cast<uint2*>(c + e) =
      make_uint2(o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16);
}

// The sum with what follows a projection in a layer: the residual added, an RMS norm of
// the row, and its largest magnitude for a conversion to fp8, as rmsnorm_kernel and
// fp8_amax_kernel have them. A row is a workgroup's, eight values a thread's, N <= 8192.
// The launches bound it, one or two less. us apart / in one, in brackets with the
// conversion: 40 rows of 1536 x 7168 13.7 / 12.1 (18.4 / 15.2), of 7168 x 16384 in fp8
// 37.9 / 35.8 (42.9 / 39.1), 96 rows of 4096 x 4096 19.4 / 17.1, 128 of 8192 x 8192 41.3
// / 38.5; the slower side nowhere from 17 rows on.
__global__ __launch_bounds__(1024) void skinny_norm_kernel(
    uint16_t* __restrict__ out, uint16_t* __restrict__ sum_out,
    uint32_t* __restrict__ largest,  // [M] or null
    const float* __restrict__ part, const uint16_t* __restrict__ residual,
    const uint16_t* __restrict__ w, const float eps, const int splits, const int M,
    const int N, const int64_t res_stride) {
  __shared__ float red[16];
  __shared__ uint32_t tops[16];
  const int row = blockIdx.x, n = threadIdx.x * 8;
  const bool on = n < N;
  float v[8], ss = 0.f;
  bf16x8 x;
  if (on) {
    const float* src = part + (size_t)row * N + n;
    const size_t all = (size_t)M * N;
    f32x4v a = {}, b = {};
#pragma unroll 8
    for (int k = 0; k < splits; ++k) {
      a += *reinterpret_cast<const f32x4v*>(src + k * all);
      b += *reinterpret_cast<const f32x4v*>(src + k * all + 4);
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const float f = r < 4 ? a[r & 3] : b[r & 3];
      v[r] = bf16_bits_to_f32(f32_to_bf16_bits(f));
    }
    if (residual != nullptr) {
      const bf16x8 rv = load_bf16x8(residual + row * res_stride + n);
#pragma unroll
      for (int r = 0; r < 8; ++r) v[r] += bf16x8_get(rv, r);
    }
    store_bf16x8(&x, v);
    if (sum_out != nullptr)
      *reinterpret_cast<int4*>(sum_out + (size_t)row * N + n) = x.raw;
#pragma unroll
    for (int r = 0; r < 8; ++r) ss = fmaf(v[r], v[r], ss);
  }
  ss = block_reduce_sum(ss, red);
  const float rstd = rsqrtf(ss / N + eps);
  uint32_t top = 0;
  if (on) {
    const bf16x8 wv = load_bf16x8(w + n);
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = bf16x8_get(x, r) * rstd * bf16x8_get(wv, r);
    store_bf16x8(&x, v);
    *reinterpret_cast<int4*>(out + (size_t)row * N + n) = x.raw;
#pragma unroll
    for (int r = 0; r < 8; ++r)
      top = max(top, __float_as_uint(bf16x8_get(x, r)) & 0x7fffffffu);
  }
  if (largest == nullptr) return;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    top = max(top, (uint32_t)__shfl_xor((int)top, o, WAVE_SIZE));
  if ((threadIdx.x & 63) == 0) tops[threadIdx.x >> 6] = top;
  __syncthreads();
  if (threadIdx.x > 0) return;
  for (int i = 1; i < (int)blockDim.x / 64; ++i) top = max(top, tops[i]);
  largest[row] = top;
}

// Waves a workgroup (32 rows of W each) and workgroups that share K: what keeps
// most of the 256 CUs busy to the end. us of 40 rows with 3 / 4 / 5 waves: 28672 x
// 4096 57 / 44 / 46, 24576 x 1536 17 / 19 / 20, 36864 x 7168 in fp8 58 / 67 / 51.
static float busy(int tiles) {
  return tiles < 256 ? tiles * (256 / tiles) / 256.f
                     : tiles / (256.f * ceil_div(tiles, 256));
}
static int skinny_waves(int N) {
  int best = 4;
  for (int w : {3, 5})
    if (busy(ceil_div(N, w * 32)) > busy(ceil_div(N, best * 32))) best = w;
  return best;
}
static int skinny_splits(int N, int row_bytes) {
  const int tiles = ceil_div(N, skinny_waves(N) * 32);
  return max(1, min(256 / tiles, min(32, row_bytes / 512)));
}

// c null: the parts alone
extern "C" void launch_skinny_split(
    void* c, float* part, int splits, const void* x, const void* w,
    const void* bias, const float* x_scale, const float* w_scale, bool fp8, int M,
    int N, int row_bytes, int64_t x_stride, int64_t c_stride, bool gated,
    hipStream_t stream) {
  const int waves = skinny_waves(N);
  auto run = [&](auto kernel) {
    const int rows = waves * (gated ? 16 : 32);
    kernel<<<dim3(ceil_div(gated ? N / 2 : N, rows), splits), waves * 64, 0,
             stream>>>(
        (uint16_t*)c, part, (const uint8_t*)x, (const uint8_t*)w,
        (const uint16_t*)bias, x_scale, w_scale, M, N, row_bytes, x_stride,
        c_stride, gated);
  };
  auto pick = [&](auto f, auto wv) {
    constexpr bool F = decltype(f)::value;
    constexpr int W = decltype(wv)::value;
    if (M <= 32) run(skinny_split_kernel<F, 1, W, 3>);
    else if (M <= 64) run(skinny_split_kernel<F, 2, W, 3>);
    else if (M <= 96) run(skinny_split_kernel<F, 3, W, W < 5 ? 4 : 3>);
    else run(skinny_split_kernel<F, 4, W, 3>);
  };
  auto by = [&](auto f) {
    if (waves == 3) pick(f, std::integral_constant<int, 3>{});
    else if (waves == 4) pick(f, std::integral_constant<int, 4>{});
    else pick(f, std::integral_constant<int, 5>{});
  };
  if (fp8) by(std::true_type{});
  else by(std::false_type{});
  if (splits > 1 && c != nullptr)
    skinny_sum_kernel<<<ceil_div(M * (gated ? N / 2 : N), 1024), 256, 0, stream>>>(
        (uint16_t*)c, part, (const uint16_t*)bias, splits, M, N, c_stride, gated);
}

extern "C" void launch_skinny_add(void* c, const float* part, const void* residual,
                                  int splits, int M, int N, int64_t res_stride,
                                  hipStream_t stream) {
  skinny_add_kernel<<<ceil_div(M * N, 1024), 256, 0, stream>>>(
      (uint16_t*)c, part, (const uint16_t*)residual, splits, M, N, res_stride);
}

extern "C" void launch_skinny_norm(void* out, void* sum_out, uint32_t* largest,
                                   const float* part, const void* residual,
                                   const void* w, float eps, int splits, int M, int N,
                                   int64_t res_stride, hipStream_t stream) {
  skinny_norm_kernel<<<M, ceil_div(N, 512) * 64, 0, stream>>>(
      (uint16_t*)out, (uint16_t*)sum_out, largest, part, (const uint16_t*)residual,
      (const uint16_t*)w, eps, splits, M, N, res_stride);
}

// Tiles, by rows of X and by how many tiles W gives. us of bf16 products, W from
// memory (N x K; the library's tuned pick last):
//   up to 8 rows, NT 8 of 8 waves / 16 of 4 where W has few rows, each CU's own rate
//   being the bound: 896 x 4864 5.7 / 6.5, 2048 x 5632 7.2 / 8.4, 1536 x 8960 8.2 /
//   11.7, 2048 x 2048 5.0 / 5.4 but 896 x 896 3.6 / 3.4, 4096 x 4096 9.2 / 8.6
//   (8 rows 6.6 / 7.5, 7.7 / 8.8, 9.7 / 11.7)
//   up to 8 rows, NT 16 of 4 waves, 5 stages / 3 stages (four workgroups a CU
//   instead of two): 28672 x 4096 40 / 41 (50), 4096 x 14336 22 / 25 (25), 9728 x
//   896 8.6 / 6.6 (12), 24576 x 1536 17 / 16 (21), 896 x 896 3.3 (5.5)
//   9 to 16, NT 16 / 32 / 64: X comes from L2 once a tile, so the widest tile
//   that still gives 150 workgroups: 6144 x 4096 14.5 / 12.1 / 16.6 (15.7),
//   28672 x 4096 48 / 45 / 42 (54), 4096 x 14336 26 / 32 / 49 (26)
//   17 to 32, the same: 28672 x 4096 60 / 47 / 43 (56), 6144 x 4096 18 / 13.9 /
//   19.5 (15.2), 4096 x 4096 10.7 / 13.4 / 19 (11.8)
static int skinny_tile(int M, int64_t N, int row_bytes, bool gated) {
  if (M <= 8) return N <= 2048 && row_bytes >= 4096 && !gated ? 8 : 16;
  if (N >= 9600) return 64;
  if (N >= 4800) return 32;
  return M <= 16 || row_bytes <= 10240 ? 16 : 0;
}

// Workgroups that share K for M rows, 0: skinny_gemm_kernel (to 32 rows), -1: the
// library. us of W alone / shared / the library: from 17 rows on where W is large
// or long, 32 rows: 24576 x 1536 19.7 / 17.2 / 21, 4096 x 14336 34 / 25 / 36, 6144 x
// 4096 13.8 / 14.8 / 16; from 9 rows on where the last tiles of 64 rows of W would
// find the CUs empty, 36864 x 7168 in fp8, 12 rows: 64 / 51 / 50. From 33 rows on:
// 28672 x 4096 at 96 rows - / 47 / 58, 4096 x 14336 - / 31 / 51; short K split, or
// small weights under many rows, cost more in parts than they gain: 9728 x 896 at 96
// rows 16 / 12, 576 x 7168 at 40 10.8 / 10.9, at 96 14 / 11. Above 128 rows: the
// library, but for the pieces below.
extern "C" int skinny_shared(int M, int N, int row_bytes) {
  if (M > 128 || row_bytes % 128 || N % 4) return -1;
  const int splits = skinny_splits(N, row_bytes);
  const int64_t bytes = (int64_t)N * row_bytes;
  if (M > 32)
    return (splits == 1 || row_bytes >= 4096) && (M <= 64 || bytes >= 1 << 24)
               ? splits : -1;
  if (M <= 8) return 0;
  const int nt = skinny_tile(M, N, row_bytes, false);
  const int tiles = ceil_div(N, 64);
  const bool ragged =
      nt == 64 && tiles > 512 && tiles < 384 * ceil_div(tiles, 512);
  return ragged || (M > 16 && (nt == 0 || bytes >= 1 << 26)) ? splits : 0;
}

// Whether a kernel above beats the library's tuned product, us of both. Short rows of
// a tall W are over before a workgroup has its copies under way; only up to 6 rows
// and from 17 to 32 do its tiles gain: 151936 x 896 with 4 / 8 / 16 / 24 / 72 / 112
// rows 52 / 55 / 59 / 57 / 73 / 85 (54 / 55 / 55 / 57 / 69 / 76), 100352 x 1024 with
// 16 / 112 46 / 65 (42 / 51); 40960 x 1024 17.7 / 24 (20 / 26) and 65536 x 2048 50 /
// 63 (67 / 77). A K split over workgroups must be long, or W large, for its parts,
// longer above 64 rows: 5120 x 2560 with 40 / 96 rows 14 / 17 (13 / 15), 3584 x 3584
// 14 / 17 (12.5 / 16), 2560 x 4096 14 / 16 (12.5 / 13), 7168 x 2048 12.5 / 15 (13 /
// 14); 4096 x 4096 12.6 / 16 (14 / 19), 1536 x 7168 12 / 14 (18 / 19). Not of the gated
// form, which saves the activation's launch besides.
extern "C" bool skinny_pays(int M, int N, int row_bytes) {
  const bool tall = N > 40960 && row_bytes < 4096;
  if (M <= 32) return !tall || M <= 6 || M > 16;
  if (skinny_splits(N, row_bytes) == 1) return !tall;
  const bool large = (int64_t)N * row_bytes >= 28000000;
  return (large || row_bytes >= 14336) && row_bytes >= (M > 64 ? 7168 : 4096);
}

// From 33 rows on, where K is not split: tiles of skinny_gemm_kernel over pieces of 32
// rows, 0: the ways above. Small weights come from L2 again for every piece, and the
// narrowest tile that still finds room on the chip at once has the shortest chain: 16
// rows of W a block while every CU has one at most, then 32 by four waves (98 KB, one
// block a CU) up to there, then 32 by two and 64 as far as two blocks a CU go. us of
// products with tiles of 16 / 32 by four waves / 32 by two / 64 rows of W and of the
// library, with its activation and bias where there are some, W from memory (N x K; gated
// ones by g, bias by b):
//   64 rows: 896 x 896 4.1 / 5.2 / 5.6 / 8.1 (6.0), 1152 x 896 b 4.4 / 5.4 / 6.1 / 9.0
//   (9.2), 2048 x 1536 b 5.2 / 6.3 / 7.6 / 11 (11), 896 x 4864 10.5 / 14 / 14 / 24 (13.3),
//   2048 x 2048 6.0 / 7.2 / 8.1 / 13 (16), and with a second round of blocks 2304 x 2048
//   8.1 / 8.3 / 8.4 / 13 (12); 3072 x 2048 9.5 / 8.5 / 8.7 / 13 (9.8), 9728 x 896 g 13 / 14 /
//   12.5 / 10.1 (14.6); in fp8 896 x 896 3.6 / - / 4.7 / 6.1 (6.1), 2048 x 8192 7.1 / 8.8 /
//   10.9 / 16 (9.4), 4096 x 7168 13 / 9.2 / 11.1 / 16 (10.1)
//   128 rows: 896 x 896 4.2 / 5.2 / 5.7 / 8.1 (6.1), 1152 x 896 b 5.6 / 5.6 / 6.1 / 9.0
//   (9.1), 2048 x 2048 8.6 / 7.3 / 8.2 / 13 (10.9), 2304 x 2048 9.6 / 10.5 / 9.0 / 13 (12),
//   896 x 4864 10.2 / 14 / 14 / 24 (13 to 21), 3072 x 3072 15 / 16 / 12.2 / 17 (16), 6144 x
//   1024 g 15 / 14 / 13 / 10.6 (12.5 to 15); in fp8 2048 x 8192 12 / 9.0 / 11 / 16 (10.5)
//   192 and 384 rows, the last: 896 x 896 5.5 / 5.3 / 5.6 / 8.1 (6.5) and 7.4 / 8.2 / 6.5 /
//   8.2 (6.6 to 8.3), 1152 x 896 b 5.9 / 5.5 / 6.1 / 9.0 (9.6) and 9.2 / 8.7 / 7.0 / 9.1
//   (12); 512: 1536 x 1536 14.4 / - / 13.6 / 12.2 (9.2)
// The lines come from 1,900 sizes drawn over 33 to 384 rows, N of 256 to 16384, rows of 512
// bytes to 16 KB, weights to 26 MB. Times as fast as the library there, in the mean and
// without the outer quarters: 16 rows 1.57 (1.36 .. 1.86), in fp8 1.82, with a bias or
// gated 1.73 to 2.00; 32 by four waves 1.31 (1.16 .. 1.44), fp8 1.44, with a bias or gated
// 1.5 to 1.7; 32 by two waves with a bias or gated, a launch less, 1.34, by themselves 1.31
// with rows of 3 KB and more, 1.15 with shorter ones, but for more than 320 blocks of up to
// 128 rows, whose tall W the library likes, 0.80 to 1.3; 64 with a bias or gated 1.17 (of
// more than 128 rows above 320 blocks 0.93 to 1.1), by themselves 0.85 (0.78 .. 0.94), in
// fp8 0.90. 16 rows go on to 384 blocks where rows of more than 8 KB leave 32 their long
// chain: 2048 x 5120 at 96 rows 14.6 / 14.4 (15.0), 2176 x 5120 16.9 / 14.8. Wide tiles have
// no time for long rows: in fp8 7168 x 2048 at 96 13 / - / 11 / 9.4 (8.9). Fewer than 64
// blocks of long rows are the library's (256 x 4096 at 40 rows 6.4 / 8.2 / 12 / 20, K split
// 8.2, library 8.9 to 11.6: a line drawn before there were pieces, and on the safe side).
// Odd widths and rows apart (linear()'s callers see to that) are torch's, whose product
// takes part in autograd and its transforms.
#define PIECES_ONE_A_CU 256
#define PIECES_MAX_M 384
#define PIECES_MAX_BYTES 26000000
static int piece_blocks(int M, int N, int nt) {
  return ceil_div(M, 32) * ceil_div(N, nt);
}
// joined: gated, or with a bias: the library's product would be followed by a launch
static int skinny_pieces(int M, int N, int row_bytes, bool gated, bool joined) {
  if (M <= 32 || M > PIECES_MAX_M || row_bytes % 128 || N % 8) return 0;
  const int64_t bytes = (int64_t)N * row_bytes;
  auto blocks = [&](int nt) { return piece_blocks(M, N, nt); };
  if (bytes > PIECES_MAX_BYTES || (row_bytes > 4096 && blocks(16) < 64)) return 0;
  if (row_bytes <= 14336 && blocks(16) <= (row_bytes > 8192 ? 384 : PIECES_ONE_A_CU))
    return 16;
  if (row_bytes <= 12288 && blocks(32) <= PIECES_ONE_A_CU) return 32;
  const int most = !joined && row_bytes < 3072 && M <= 128 ? 320
                   : bytes > 20000000 ? 340 : 384;
  if (row_bytes <= (N > 2048 ? 12288 : 6144) && blocks(32) <= most) return 32;
  return joined && row_bytes <= (gated ? 2048 : 1920) &&
                 blocks(64) <= (M > 128 ? 320 : 512)
             ? 64 : 0;
}

// The rows and bytes of W above which there are none: callers that must not wait for the
// rule ask these first.
extern "C" void skinny_pieces_limits(int* rows, int64_t* bytes) {
  *rows = PIECES_MAX_M;
  *bytes = PIECES_MAX_BYTES;
}

// K split over workgroups stays: its parts are what launch_skinny_norm adds up
extern "C" bool skinny_in_pieces(int M, int N, int row_bytes, bool gated, bool bias) {
  return skinny_pieces(M, N, row_bytes, gated, gated || bias) > 0 &&
         (skinny_shared(M, N, row_bytes) <= 1 ||
          (!gated && !skinny_pays(M, N, row_bytes)));
}

// batch products of the same shape: x, w and c advance by x_batch bytes, N rows
// and c_batch elements. Any number of rows of X, 32 at a time.
extern "C" void launch_skinny_gemm(
    void* c, const void* x, const void* w, const void* bias,
    const float* x_scale, const float* w_scale, bool fp8, int M, int N,
    int row_bytes, int64_t x_stride, int64_t c_stride, int batch,
    int64_t x_batch, int64_t c_batch, bool gated, hipStream_t stream,
    bool* launched) {
  *launched = false;
  int nt = batch == 1 ? skinny_pieces(M, N, row_bytes, gated, gated || bias != nullptr)
                      : 0;
  if (nt == 0) nt = skinny_tile(min(M, 32), (int64_t)N * batch, row_bytes, gated);
  if (nt == 0 || row_bytes % 128 || N % 4) return;
  *launched = true;
  auto run = [&](auto kernel, int xr, int waves) {
    const int tiles = gated ? ceil_div(N / 2, nt / 2) : ceil_div(N, nt);
    kernel<<<dim3(tiles, batch, ceil_div(M, xr)), waves * 64, 0, stream>>>(
        (uint16_t*)c, (const uint8_t*)x, (const uint8_t*)w,
        (const uint16_t*)bias, x_scale, w_scale, M, N, row_bytes, x_stride,
        c_stride, x_batch, c_batch, gated);
  };
  auto pick = [&](auto f) {
    constexpr bool F = decltype(f)::value;
    if (M <= 8) {
      if (nt == 8) run(skinny_gemm_kernel<F, 8, 8, 8, 4>, 8, 8);
      else if (row_bytes <= 4096) run(skinny_gemm_kernel<F, 16, 8, 4, 3>, 8, 4);
      else run(skinny_gemm_kernel<F, 16, 8, 4, 5>, 8, 4);
    } else if (M <= 16) {
      if (nt == 64) run(skinny_gemm_kernel<F, 64, 16, 2, 4>, 16, 2);
      else if (nt == 32) run(skinny_gemm_kernel<F, 32, 16, 4, 3>, 16, 4);
      else run(skinny_gemm_kernel<F, 16, 16, 4, 4>, 16, 4);
    } else {
      if (nt == 64) run(skinny_gemm_kernel<F, 64, 32, 2, 3>, 32, 2);
      else if (nt == 32 && M > 32 && batch == 1 &&
               piece_blocks(M, N, 32) <= PIECES_ONE_A_CU)
        run(skinny_gemm_kernel<F, 32, 32, 4, 3>, 32, 4);
      else if (nt == 32) run(skinny_gemm_kernel<F, 32, 32, 2, 4>, 32, 2);
      else run(skinny_gemm_kernel<F, 16, 32, 4, 3>, 32, 4);
    }
  };
  if (fp8) pick(std::true_type{});
  else pick(std::false_type{});
}

// ---- MLA queries into latent space ----------------------------------------------------
// out[b, h] = q[b, h] . W[h] of [128, R]: rows of W run along the result, so its
// operand is read transposed from LDS. A workgroup takes 128 of the R columns of
// one head and 32 rows of q, one pass. W's stream bounds it: 40 rows at 128
// heads 9 us, fp32 copies and an fp32
// product before 45 us.

__global__ __launch_bounds__(256) void mla_absorb_kernel(
    uint16_t* __restrict__ out,      // [B, H, R]
    const uint16_t* __restrict__ q,  // [B, H, 128] by strides
    const uint16_t* __restrict__ w,  // [H, 128, R]
    const int B, const int H, const int R, const int64_t q_row,
    const int64_t q_head) {
  __shared__ __attribute__((aligned(128))) uint16_t W[128 * 128];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, l31 = lane & 31;
  const int h = blockIdx.y;
  const int b = blockIdx.z * 32 + l31;
  const uint16_t* src = w + (size_t)h * 128 * R + blockIdx.x * 128;
  // 16-byte chunk j of row k lies at j ^ 4 (k & 3)
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int k = i * 16 + (tid >> 4);
    copy16_to_lds(src + (size_t)k * R + ((tid & 15) ^ ((k & 3) * 4)) * 8,
                  W + (i * 16 + wid * 4) * 128);
  }
  bf16x8v x[8];
  const uint16_t* qr =
      q + (size_t)min(b, B - 1) * q_row + (size_t)h * q_head + half * 8;
#pragma unroll
  for (int s = 0; s < 8; ++s) x[s] = *(const bf16x8v*)(qr + s * 16);
  wait_copies<0>();
  __syncthreads();
  const int i15 = lane & 15;
  const int chunk = (wid * 4 + ((lane >> 4) & 1) * 2 + ((i15 & 3) >> 1)) ^
                    ((i15 >> 2) * 4);
  uint16_t* at = W + (half * 8 + (i15 >> 2)) * 128 + chunk * 8 + (i15 & 1) * 4;
  f32x16v acc = {};
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const s16x4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4v*)(at + s * 16 * 128));
    const s16x4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4v*)(at + s * 16 * 128 + 4 * 128));
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), x[s], acc, 0, 0,
        0);
  }
  if (b >= B) return;
  uint16_t* dst = out + ((size_t)b * H + h) * R + blockIdx.x * 128 + wid * 32 +
                  4 * half;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint16_t o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = f32_to_bf16_bits(acc[4 * i + r]);
    *reinterpret_cast<uint2*>(dst + 8 * i) =
        make_uint2(o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16);
  }
}

extern "C" void launch_mla_absorb(void* out, const void* q, const void* w, int B,
                                  int H, int R, int64_t q_row, int64_t q_head,
                                  hipStream_t stream) {
  mla_absorb_kernel<<<dim3(R / 128, H, ceil_div(B, 32)), 256, 0, stream>>>(
      (uint16_t*)out, (const uint16_t*)q, (const uint16_t*)w, B, H, R, q_row,
      q_head);
}

// ---- activations to fp8 (OCP e4m3), one scale a tensor -------------------------------
// scale = max(amax * (1 / 448), 1e-8), values x / scale clamped to +-448. Two passes:
// the largest magnitude a workgroup (as bits, so that NaN is the largest), then
// every workgroup reduces those and converts its part. Launches bound it at
// decode sizes: 2 instead of 7 operations of torch and a copy. From some 500,000 values
// on it is the loads in flight, so the grids grow until the chip is full: both launches
// with at most 256 workgroups each / with 1,024 and 2,048: 700 x 7168 12.0 / 10.0 us,
// 700 x 18432 23.8 / 17.3, 2,500 x 18432 85.0 / 48.9 (2 x 92 MB read and
// 46 written take 38 at 6.1 TB/s); 300 x 7168 and fewer the same within 2%.

#define Q8_MAX_BLOCKS 1024   // of the first pass

template <typename T>
DEVINL uint32_t magnitude(T v) {
  if constexpr (sizeof(T) == 2) return (uint32_t)(v & 0x7fff) << 16;
  else return v & 0x7fffffffu;
}

DEVINL uint32_t block_max(uint32_t m, uint32_t* lds) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, 64));
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = m;
  __syncthreads();
  return max(max(lds[0], lds[1]), max(lds[2], lds[3]));
}

// T: the bits of a bf16 or fp32 value; whole vectors of 8 first, then the rest
template <typename T, typename F>
DEVINL void for_each8(const T* x, int64_t n, bool aligned, F f) {
  struct __attribute__((aligned(16))) V { T v[8]; };
  const int64_t step = (int64_t)gridDim.x * 256;
  const int64_t first = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t nv = aligned ? n / 8 : 0;
  for (int64_t i = first; i < nv; i += step) {
    const V v = reinterpret_cast<const V*>(x)[i];
    f(i * 8, v.v, 8);
  }
  for (int64_t i = nv * 8 + first; i < n; i += step) f(i, x + i, 1);
}

template <typename T>
__global__ __launch_bounds__(256) void fp8_amax_kernel(
    uint32_t* __restrict__ part, const T* __restrict__ x, const int64_t n,
    const bool aligned) {
  __shared__ uint32_t lds[4];
  uint32_t m = 0;
  for_each8(x, n, aligned, [&](int64_t, const T* v, int c) {
    for (int j = 0; j < c; ++j) m = max(m, magnitude(v[j]));
  });
  m = block_max(m, lds);
  if (threadIdx.x == 0) part[blockIdx.x] = m;
}

template <typename T>
__global__ __launch_bounds__(256) void fp8_convert_kernel(
    uint8_t* __restrict__ out, float* __restrict__ scale_out,
    const uint32_t* __restrict__ part, const T* __restrict__ x, const int64_t n,
    const bool aligned, const int parts) {
  __shared__ uint32_t lds[4];
  uint32_t m = 0;
  for (int i = threadIdx.x; i < parts; i += 256) m = max(m, part[i]);
  float scale = __uint_as_float(block_max(m, lds)) * (1.f / 448.f);
  if (scale < 1e-8f) scale = 1e-8f;
  if (blockIdx.x == 0 && threadIdx.x == 0) *scale_out = scale;
  for_each8(x, n, aligned, [&](int64_t i, const T* v, int c) {
    uint64_t q = 0;
    for (int j = 0; j < c; ++j) {
      float f = (sizeof(T) == 2 ? __uint_as_float((uint32_t)v[j] << 16)
                                : __uint_as_float((uint32_t)v[j])) / scale;
      f = f > 448.f ? 448.f : f < -448.f ? -448.f : f;
      q |= (uint64_t)f32_to_fp8_e4m3(f) << (8 * j);
    }
    if (c == 8) *reinterpret_cast<uint64_t*>(out + i) = q;
    else out[i] = (uint8_t)q;
  });
}

extern "C" int quantize_fp8_tensor_parts(int64_t n) {
  return clamp_int((n + 2047) / 2048, 1, Q8_MAX_BLOCKS);
}

// parts > 0: the largest magnitudes of that many parts of x are in part already
extern "C" void launch_quantize_fp8_tensor(void* out, float* scale,
                                           uint32_t* part, const void* x,
                                           int64_t n, bool is_bf16, int parts,
                                           hipStream_t stream) {
  const int blocks = quantize_fp8_tensor_parts(n);
  const bool aligned = (uintptr_t)x % 16 == 0 && (uintptr_t)out % 8 == 0;
  auto run = [&](auto* p) {
    if (parts == 0)
      fp8_amax_kernel<<<blocks, 256, 0, stream>>>(part, p, n, aligned);
    fp8_convert_kernel<<<clamp_int((n + 2047) / 2048, 1, 2048), 256, 0, stream>>>(
        (uint8_t*)out, scale, part, p, n, aligned, parts == 0 ? blocks : parts);
  };
  if (is_bf16) run((const uint16_t*)x);
  else run((const uint32_t*)x);
}
