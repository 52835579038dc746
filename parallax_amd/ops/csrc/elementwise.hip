// Memory-bound elementwise / normalization kernels for gfx950.
// All bf16 traffic is vectorized 16 B/lane (bf16x8) per the CDNA guide (G13).
//
// Reference analogues: RMSNorm/RoPE/activation live inside MLX / SGLang in the
// reference; here they are first-class HIP kernels fused where it pays
// (fused_add_rmsnorm saves two HBM round-trips per layer).

#include <type_traits>

#include "common.h"

// ---- rmsnorm -------------------------------------------------------------------
// x: [rows, H] bf16, w: [H] bf16, out: [rows, H]. One block per row.
// fp32 accumulation; H must be a multiple of 8.

template <bool FUSED_ADD>
__global__ void rmsnorm_kernel(
    uint16_t* __restrict__ out,          // [rows, H] (bf16 bits)
    uint16_t* __restrict__ x,            // [rows, H] — input; mutated if FUSED_ADD
    uint16_t* __restrict__ residual,     // [rows, H] or nullptr
    const uint16_t* __restrict__ w,      // [H]
    const float eps,
    const int H) {
  __shared__ float red[16];
  const int row = blockIdx.x;
  uint16_t* xr = x + (size_t)row * H;
  uint16_t* rr = FUSED_ADD ? residual + (size_t)row * H : nullptr;
  uint16_t* orow = out + (size_t)row * H;

  const int vecs = H / 8;
  float ss = 0.f;
  // pass 1: (optional add) + sum of squares; FUSED_ADD writes the new residual
  for (int i = threadIdx.x; i < vecs; i += blockDim.x) {
    bf16x8 xv = load_bf16x8(xr + i * 8);
    float vals[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) vals[j] = bf16x8_get(xv, j);
    if (FUSED_ADD) {
      bf16x8 rv = load_bf16x8(rr + i * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) vals[j] += bf16x8_get(rv, j);
      store_bf16x8(rr + i * 8, vals);  // residual' = x + residual
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) ss = fmaf(vals[j], vals[j], ss);
  }
  ss = block_reduce_sum(ss, red);
  const float rstd = rsqrtf(ss / H + eps);
  __syncthreads();

  // pass 2: normalize * weight  (rows are L2-resident between passes)
  const uint16_t* src = FUSED_ADD ? rr : xr;
  for (int i = threadIdx.x; i < vecs; i += blockDim.x) {
    bf16x8 xv = load_bf16x8(src + i * 8);
    bf16x8 wv = load_bf16x8(w + i * 8);
    float vals[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      vals[j] = bf16x8_get(xv, j) * rstd * bf16x8_get(wv, j);
    store_bf16x8(orow + i * 8, vals);
  }
}

extern "C" void launch_rmsnorm(
    void* out, void* x, const void* w, float eps, int rows, int H,
    hipStream_t stream) {
  int threads = min(1024, max(64, ((H / 8) + 63) / 64 * 64));
  rmsnorm_kernel<false><<<rows, threads, 0, stream>>>(
      (uint16_t*)out, (uint16_t*)x, nullptr, (const uint16_t*)w, eps, H);
}

extern "C" void launch_fused_add_rmsnorm(
    void* x, void* residual, const void* w, float eps, int rows, int H,
    hipStream_t stream) {
  int threads = min(1024, max(64, ((H / 8) + 63) / 64 * 64));
  // out == x (in-place): x <- rmsnorm(x + residual), residual <- x + residual
  rmsnorm_kernel<true><<<rows, threads, 0, stream>>>(
      (uint16_t*)x, (uint16_t*)x, (uint16_t*)residual, (const uint16_t*)w, eps, H);
}

// ---- RoPE (neox + interleaved) ---------------------------------------------------
// q: [T, Hq, D], k: [T, Hk, D] (bf16, mutated in place), positions: [T] i32,
// cos_sin: [P, rot] fp32 (cos | sin halves). Host-precomputed table (guide §B).
// One block per token; threads sweep (head, pair).

template <bool NEOX>
__global__ void rope_kernel(
    uint16_t* __restrict__ q, uint16_t* __restrict__ k,
    const int* __restrict__ positions, const float* __restrict__ cos_sin,
    const int Hq, const int Hk, const int D, const int rot,
    const int64_t q_stride, const int64_t k_stride) {
  const int t = blockIdx.x;
  const int half = rot / 2;
  const float* cs = cos_sin + (size_t)positions[t] * rot;
  const int total = (Hq + Hk) * half;
  for (int i = threadIdx.x; i < total; i += blockDim.x) {
    const int h = i / half;
    const int j = i % half;
    uint16_t* base = (h < Hq) ? q + (size_t)t * q_stride + h * D
                              : k + (size_t)t * k_stride + (h - Hq) * D;
    const float c = cs[j], s = cs[half + j];
    int i1, i2;
    if (NEOX) {
      i1 = j; i2 = j + half;
    } else {
      i1 = 2 * j; i2 = 2 * j + 1;
    }
    const float x1 = bf16_bits_to_f32(base[i1]);
    const float x2 = bf16_bits_to_f32(base[i2]);
    base[i1] = f32_to_bf16_bits(fmaf(x1, c, -x2 * s));
    base[i2] = f32_to_bf16_bits(fmaf(x2, c, x1 * s));
  }
}

extern "C" void launch_rope(
    void* q, void* k, const int* positions, const float* cos_sin,
    int T, int Hq, int Hk, int D, int rot, bool neox, int64_t q_stride,
    int64_t k_stride, hipStream_t stream) {
  int threads = min(512, max(64, ceil_div((Hq + Hk) * rot / 2, 64) * 64));
  if (neox)
    rope_kernel<true><<<T, threads, 0, stream>>>(
        (uint16_t*)q, (uint16_t*)k, positions, cos_sin, Hq, Hk, D, rot,
        q_stride, k_stride);
  else
    rope_kernel<false><<<T, threads, 0, stream>>>(
        (uint16_t*)q, (uint16_t*)k, positions, cos_sin, Hq, Hk, D, rot,
        q_stride, k_stride);
}

// ---- fused rope + cache scatter ----------------------------------------------------
// One launch per decode/prefill step replaces {rope(q,k) ; reshape_and_cache}:
// q roped in place (strided rows OK), k roped straight into the paged cache,
// v copied vectorized. Saves one k round-trip and two kernel launches per layer.
template <bool NEOX, bool FP8>
__global__ void rope_and_cache_kernel(
    uint16_t* __restrict__ q,        // [T, Hq, D] rows at q_stride
    const uint16_t* __restrict__ k,  // [T, Hk, D] rows at k_stride
    const uint16_t* __restrict__ v,
    void* __restrict__ k_cache_v,    // [NB, Hk, BS, D] bf16 | fp8
    void* __restrict__ v_cache_v,
    const int* __restrict__ positions, const float* __restrict__ cos_sin,
    const int64_t* __restrict__ slot_mapping,
    const int Hq, const int Hk, const int D, const int rot, const int BS,
    const int64_t q_stride, const int64_t k_stride, const int64_t v_stride,
    const float inv_k_scale, const float inv_v_scale) {
  const int t = blockIdx.x;
  const int64_t slot = slot_mapping[t];
  const int half = rot / 2;
  const float* cs = cos_sin + (size_t)positions[t] * rot;
  const int64_t blk = slot >= 0 ? slot / BS : 0;
  const int64_t off = slot >= 0 ? slot % BS : 0;
  const size_t base_off = (((size_t)blk * Hk) * BS + off) * D;
  // v cache is transposed [NB, Hk, D, BS]: per-(h,d) element lands at column
  // `off` of the d row
  const size_t vbase_off = ((size_t)blk * Hk) * (size_t)D * BS + off;
  uint16_t* kdst16 = FP8 ? nullptr : (uint16_t*)k_cache_v + base_off;
  uint16_t* vdst16 = FP8 ? nullptr : (uint16_t*)v_cache_v + vbase_off;
  uint8_t* kdst8 = FP8 ? (uint8_t*)k_cache_v + base_off : nullptr;
  uint8_t* vdst8 = FP8 ? (uint8_t*)v_cache_v + vbase_off : nullptr;

  // q: rope in place
  for (int i = threadIdx.x; i < Hq * half; i += blockDim.x) {
    const int h = i / half, j = i % half;
    uint16_t* base = q + (size_t)t * q_stride + h * D;
    const float c = cs[j], ss = cs[half + j];
    const int i1 = NEOX ? j : 2 * j;
    const int i2 = NEOX ? j + half : 2 * j + 1;
    const float x1 = bf16_bits_to_f32(base[i1]);
    const float x2 = bf16_bits_to_f32(base[i2]);
    base[i1] = f32_to_bf16_bits(fmaf(x1, c, -x2 * ss));
    base[i2] = f32_to_bf16_bits(fmaf(x2, c, x1 * ss));
  }
  if (slot < 0) return;
  // k: rope -> cache (rot dims) + copy (pass-through dims if rot < D)
  for (int i = threadIdx.x; i < Hk * half; i += blockDim.x) {
    const int h = i / half, j = i % half;
    const uint16_t* src = k + (size_t)t * k_stride + h * D;
    const float c = cs[j], ss = cs[half + j];
    const int i1 = NEOX ? j : 2 * j;
    const int i2 = NEOX ? j + half : 2 * j + 1;
    const float x1 = bf16_bits_to_f32(src[i1]);
    const float x2 = bf16_bits_to_f32(src[i2]);
    const float o1 = fmaf(x1, c, -x2 * ss);
    const float o2 = fmaf(x2, c, x1 * ss);
    if (FP8) {
      kdst8[(size_t)h * BS * D + i1] = f32_to_fp8_e4m3(o1 * inv_k_scale);
      kdst8[(size_t)h * BS * D + i2] = f32_to_fp8_e4m3(o2 * inv_k_scale);
    } else {
      kdst16[(size_t)h * BS * D + i1] = f32_to_bf16_bits(o1);
      kdst16[(size_t)h * BS * D + i2] = f32_to_bf16_bits(o2);
    }
  }
  if (rot < D) {
    for (int i = threadIdx.x; i < Hk * (D - rot); i += blockDim.x) {
      const int h = i / (D - rot);
      const int d = rot + i % (D - rot);
      const float x = bf16_bits_to_f32(k[(size_t)t * k_stride + h * D + d]);
      if (FP8)
        kdst8[(size_t)h * BS * D + d] = f32_to_fp8_e4m3(x * inv_k_scale);
      else
        kdst16[(size_t)h * BS * D + d] = f32_to_bf16_bits(x);
    }
  }
  // v: transpose-scatter into the [.., D, BS] layout (quantized when FP8) —
  // one 2 B store per element at decode (1 token); the attention kernels'
  // fragment loads read V^T contiguously in exchange
  for (int i = threadIdx.x; i < Hk * D; i += blockDim.x) {
    const int h = i / D;
    const int d = i % D;
    const float x = bf16_bits_to_f32(v[(size_t)t * v_stride + h * D + d]);
    const size_t dst = ((size_t)h * D + d) * BS;
    if (FP8)
      vdst8[dst] = f32_to_fp8_e4m3(x * inv_v_scale);
    else
      vdst16[dst] = f32_to_bf16_bits(x);
  }
}

// The same, 16 elements a thread. Bound by memory at prefill, 8,192 tokens of 32
// and 8 heads of 128 52 us or 3.9 TB/s, 57 us from an odd slot (value by value 115);
// by latency at decode, 96 tokens 4.7 us (9.3: one workgroup a token). The first
// rope_blocks take a rotated or copied piece of q or k a thread, the others 8 values
// of one v head; with RUNS eight tokens' at once where their slots are neighbours.
template <bool NEOX, bool FP8, bool RUNS>
__global__ __launch_bounds__(256) void rope_and_cache8_kernel(
    uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, void* __restrict__ k_cache,
    void* __restrict__ v_cache, const int* __restrict__ positions,
    const float* __restrict__ cos_sin, const int64_t* __restrict__ slot_mapping,
    const int T, const int Hq, const int Hk, const int D, const int rot,
    const int BS, const int64_t q_stride, const int64_t k_stride,
    const int64_t v_stride, const float inv_k_scale, const float inv_v_scale,
    const int rope_blocks) {
  using C = std::conditional_t<FP8, uint8_t, uint16_t>;
  auto store8 = [](C* dst, const float* x, float inv) {
    if constexpr (FP8) {
      uint64_t o = 0;
#pragma unroll
      for (int r = 0; r < 8; ++r)
        o |= (uint64_t)f32_to_fp8_e4m3(x[r] * inv) << (8 * r);
      *reinterpret_cast<uint64_t*>(dst) = o;
    } else {
      store_bf16x8(dst, x);
    }
  };
  if ((int)blockIdx.x < rope_blocks) {
    const int half = rot / 2;
    const int turns = half / 8;                  // rotated pieces a head
    const int k_items = turns + (D - rot) / 8;   // and copied ones of k
    const int per_token = Hq * turns + Hk * k_items;
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int t = (int)(e / per_token);
    if (t >= T) return;
    int i = (int)(e % per_token);
    const bool is_q = i < Hq * turns;
    if (!is_q) i -= Hq * turns;
    const int h = i / (is_q ? turns : k_items);
    const int piece = i % (is_q ? turns : k_items);
    C* kd = nullptr;
    if (!is_q) {
      const int64_t slot = slot_mapping[t];
      if (slot < 0) return;
      kd = (C*)k_cache + (((slot / BS) * Hk + h) * BS + slot % BS) * D;
    }
    if (piece >= turns) {
      const int d = rot + (piece - turns) * 8;
      const bf16x8 x = load_bf16x8(k + (int64_t)t * k_stride + h * D + d);
      float f[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) f[r] = bf16x8_get(x, r);
      store8(kd + d, f, inv_k_scale);
      return;
    }
    const int j = piece * 8;
    const float* cs = cos_sin + (size_t)positions[t] * rot + j;
    float c[8], ss[8];
#pragma unroll
    for (int r = 0; r < 8; r += 4) {
      *reinterpret_cast<f32x4v*>(c + r) = *reinterpret_cast<const f32x4v*>(cs + r);
      *reinterpret_cast<f32x4v*>(ss + r) =
          *reinterpret_cast<const f32x4v*>(cs + half + r);
    }
    const int i1 = NEOX ? j : 2 * j, i2 = NEOX ? j + half : 2 * j + 8;
    const uint16_t* src = is_q ? q + (int64_t)t * q_stride + h * D
                               : k + (int64_t)t * k_stride + h * D;
    const bf16x8 a = load_bf16x8(src + i1), b = load_bf16x8(src + i2);
    float x[16], o[16];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      x[r] = bf16x8_get(a, r);
      x[8 + r] = bf16x8_get(b, r);
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int n1 = NEOX ? r : 2 * r, n2 = NEOX ? 8 + r : 2 * r + 1;
      o[n1] = fmaf(x[n1], c[r], -x[n2] * ss[r]);
      o[n2] = fmaf(x[n2], c[r], x[n1] * ss[r]);
    }
    if (is_q) {
      uint16_t* dst = q + (int64_t)t * q_stride + h * D;
      store_bf16x8(dst + i1, o);
      store_bf16x8(dst + i2, o + 8);
    } else {
      store8(kd + i1, o, inv_k_scale);
      store8(kd + i2, o + 8, inv_k_scale);
    }
    return;
  }
  // ---- v -----------------------------------------------------------------------------
  const int per_token = Hk * D / 8;
  auto row = [&](int64_t slot, int h, int d) {
    return (C*)v_cache + (((slot / BS) * Hk + h) * D + d) * BS + slot % BS;
  };
  auto put = [&](int t, int64_t slot, int h, int d) {
    const bf16x8 x = load_bf16x8(v + (int64_t)t * v_stride + h * D + d);
    C* dst = row(slot, h, d);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const float f = bf16x8_get(x, r);
      if constexpr (FP8) dst[r * BS] = f32_to_fp8_e4m3(f * inv_v_scale);
      else dst[r * BS] = f32_to_bf16_bits(f);
    }
  };
  if constexpr (!RUNS) {
    const int64_t e = (int64_t)(blockIdx.x - rope_blocks) * 256 + threadIdx.x;
    const int t = (int)(e / per_token), i = (int)(e % per_token) * 8;
    if (t >= T || slot_mapping[t] < 0) return;
    put(t, slot_mapping[t], i / D, i % D);
  } else {
    // A wave has the tokens t0 .. t0 + 7 and 64 items of each. Eight neighbouring
    // slots from a multiple of 8 on are stored at once by the wave in whose eight
    // tokens they begin; what lies in no such run goes by itself.
    const int lane = threadIdx.x & 63;
    const int chunks = (per_token + 63) / 64;
    const int64_t wave =
        (int64_t)(blockIdx.x - rope_blocks) * 4 + (threadIdx.x >> 6);
    const int t0 = (int)(wave / chunks) * 8;
    if (t0 >= T) return;
    const int near = t0 - 8 + lane;  // lanes 8 .. 15: this wave's tokens
    const int64_t slot =
        lane < 24 && near >= 0 && near < T ? slot_mapping[near] : -1;
    const bool next = slot >= 0 && __shfl_down(slot, 1, WAVE_SIZE) == slot + 1;
    const unsigned long long runs = __ballot(next);
    const unsigned long long begins =
        __ballot(slot >= 0 && slot % 8 == 0 && BS % 8 == 0 &&
                 ((runs >> lane) & 0x7f) == 0x7f);
    const int before = begins & 0xff ? __ffsll(begins & 0xff) - 1 : 0;
    const int here = (begins >> 8) & 0xff ? __ffsll((begins >> 8) & 0xff) - 1 : 8;
    const int item = (int)(wave % chunks) * 64 + lane;
    const bool on = item < per_token;
    const int h = item * 8 / D, d = item * 8 % D;
    for (int i = before; i < here; ++i) {
      const int64_t s = __shfl(slot, 8 + i, WAVE_SIZE);
      if (on && s >= 0) put(t0 + i, s, h, d);
    }
    if (here == 8) return;
    const int64_t s0 = __shfl(slot, 8 + here, WAVE_SIZE);
    if (!on) return;
    C val[8][8];  // [d][token]
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bf16x8 x =
          load_bf16x8(v + (int64_t)(t0 + here + i) * v_stride + h * D + d);
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const float f = bf16x8_get(x, r);
        if constexpr (FP8) val[r][i] = f32_to_fp8_e4m3(f * inv_v_scale);
        else val[r][i] = f32_to_bf16_bits(f);
      }
    }
    using V = std::conditional_t<FP8, uint2, uint4>;
    C* dst = row(s0, h, d);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      V o;
      __builtin_memcpy(&o, val[r], sizeof(V));
      *reinterpret_cast<V*>(dst + r * BS) = o;
    }
  }
}

extern "C" void launch_rope_and_cache(
    void* q, const void* k, const void* v, void* k_cache, void* v_cache,
    const int* positions, const float* cos_sin, const int64_t* slot_mapping,
    int T, int Hq, int Hk, int D, int rot, int BS, bool neox, bool fp8,
    float k_scale, float v_scale, int64_t q_stride, int64_t k_stride,
    int64_t v_stride, hipStream_t stream) {
  const float iks = 1.f / k_scale, ivs = 1.f / v_scale;
  uintptr_t at = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v |
                 (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)cos_sin;
  if (rot % 16 == 0 && D % 8 == 0 && at % 16 == 0 &&
      (q_stride | k_stride | v_stride) % 8 == 0) {
    if (T == 0) return;
    // runs of slots for prompts: 1,024 tokens 7.9 us, a token a thread 12.2; 96
    // requests, a slot each, 12.2 and 4.7
    const bool runs = T >= 1024;
    const int64_t per_token =
        (int64_t)Hq * (rot / 16) + (int64_t)Hk * (rot / 16 + (D - rot) / 8);
    const int rope_blocks = (int)ceil_div(T * per_token, 256);
    const int items = Hk * D / 8;
    const int blocks =
        rope_blocks + (runs ? ceil_div(ceil_div(T, 8) * ceil_div(items, 64), 4)
                            : ceil_div(T * items, 256));
    auto run = [&](auto kernel) {
      kernel<<<blocks, 256, 0, stream>>>(
          (uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, k_cache, v_cache,
          positions, cos_sin, slot_mapping, T, Hq, Hk, D, rot, BS, q_stride,
          k_stride, v_stride, iks, ivs, rope_blocks);
    };
    auto pick = [&](auto n, auto f) {
      constexpr bool N = decltype(n)::value, F = decltype(f)::value;
      if (runs) run(rope_and_cache8_kernel<N, F, true>);
      else run(rope_and_cache8_kernel<N, F, false>);
    };
    if (neox && fp8) pick(std::true_type{}, std::true_type{});
    else if (neox) pick(std::true_type{}, std::false_type{});
    else if (fp8) pick(std::false_type{}, std::true_type{});
    else pick(std::false_type{}, std::false_type{});
    return;
  }
  int threads = min(512, max(128, ceil_div(Hk * D / 8, 64) * 64));
#define RC_LAUNCH(NEOX, FP8)                                                 \
  rope_and_cache_kernel<NEOX, FP8><<<T, threads, 0, stream>>>(              \
      (uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, k_cache,        \
      v_cache, positions, cos_sin, slot_mapping, Hq, Hk, D, rot, BS,        \
      q_stride, k_stride, v_stride, iks, ivs)
  if (neox && fp8) RC_LAUNCH(true, true);
  else if (neox) RC_LAUNCH(true, false);
  else if (fp8) RC_LAUNCH(false, true);
  else RC_LAUNCH(false, false);
#undef RC_LAUNCH
}

// ---- reshape_and_cache ------------------------------------------------------------
// k/v: [T, Hk, D] bf16 -> k_cache/v_cache [NB, Hk, BS, D] via slot_mapping [T]
// (slot = block * BS + off; -1 skips). One block per token, vectorized rows.

__global__ void reshape_and_cache_kernel(
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    uint16_t* __restrict__ k_cache, uint16_t* __restrict__ v_cache,
    const int64_t* __restrict__ slot_mapping,
    const int Hk, const int D, const int BS) {
  const int t = blockIdx.x;
  const int64_t slot = slot_mapping[t];
  if (slot < 0) return;
  const int64_t blk = slot / BS, off = slot % BS;
  const int vecs = Hk * D / 8;
  const uint16_t* ksrc = k + (size_t)t * Hk * D;
  const uint16_t* vsrc = v + (size_t)t * Hk * D;
  for (int i = threadIdx.x; i < vecs; i += blockDim.x) {
    const int h = (i * 8) / D;
    const int d = (i * 8) % D;
    // k row: cache[blk][h][off][d]
    const size_t dst = (((size_t)blk * Hk + h) * BS + off) * D + d;
    *reinterpret_cast<int4*>(k_cache + dst) =
        *reinterpret_cast<const int4*>(ksrc + i * 8);
    // v transposed: cache[blk][h][d + j][off]
    const int4 vv = *reinterpret_cast<const int4*>(vsrc + i * 8);
    const uint16_t* ve = reinterpret_cast<const uint16_t*>(&vv);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v_cache[(((size_t)blk * Hk + h) * D + d + j) * BS + off] = ve[j];
  }
}

extern "C" void launch_reshape_and_cache(
    const void* k, const void* v, void* k_cache, void* v_cache,
    const int64_t* slot_mapping, int T, int Hk, int D, int BS,
    hipStream_t stream) {
  int threads = min(512, max(64, ceil_div(Hk * D / 8, 64) * 64));
  reshape_and_cache_kernel<<<T, threads, 0, stream>>>(
      (const uint16_t*)k, (const uint16_t*)v, (uint16_t*)k_cache,
      (uint16_t*)v_cache, slot_mapping, Hk, D, BS);
}

// MLA variant: latent [T, R] + rope [T, dr] -> cache [NB, BS, R+dr]
template <bool FP8>
__global__ void mla_reshape_and_cache_kernel(
    const uint16_t* __restrict__ latent, const uint16_t* __restrict__ k_rope,
    void* __restrict__ cache, const int64_t* __restrict__ slot_mapping,
    const int R, const int DR, const int BS, const float inv_scale) {
  const int t = blockIdx.x;
  const int64_t slot = slot_mapping[t];
  if (slot < 0) return;
  const int64_t blk = slot / BS, off = slot % BS;
  const size_t row = ((size_t)blk * BS + off) * (R + DR);
  if (FP8) {
    uint8_t* dst = (uint8_t*)cache + row;
    for (int i = threadIdx.x * 8; i < R; i += blockDim.x * 8) {
      uint64_t packed = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        packed |= (uint64_t)f32_to_fp8_e4m3(
                      bf16_bits_to_f32(latent[(size_t)t * R + i + j]) *
                      inv_scale)
                  << (8 * j);
      *reinterpret_cast<uint64_t*>(dst + i) = packed;
    }
    for (int i = threadIdx.x * 8; i < DR; i += blockDim.x * 8) {
      uint64_t packed = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        packed |= (uint64_t)f32_to_fp8_e4m3(
                      bf16_bits_to_f32(k_rope[(size_t)t * DR + i + j]) *
                      inv_scale)
                  << (8 * j);
      *reinterpret_cast<uint64_t*>(dst + R + i) = packed;
    }
  } else {
    uint16_t* dst = (uint16_t*)cache + row;
    for (int i = threadIdx.x * 8; i < R; i += blockDim.x * 8)
      *reinterpret_cast<int4*>(dst + i) =
          *reinterpret_cast<const int4*>(latent + (size_t)t * R + i);
    for (int i = threadIdx.x * 8; i < DR; i += blockDim.x * 8)
      *reinterpret_cast<int4*>(dst + R + i) =
          *reinterpret_cast<const int4*>(k_rope + (size_t)t * DR + i);
  }
}

extern "C" void launch_mla_reshape_and_cache(
    const void* latent, const void* k_rope, void* cache,
    const int64_t* slot_mapping, int T, int R, int DR, int BS, bool fp8,
    float inv_scale, hipStream_t stream) {
  if (fp8)
    mla_reshape_and_cache_kernel<true><<<T, 128, 0, stream>>>(
        (const uint16_t*)latent, (const uint16_t*)k_rope, cache, slot_mapping,
        R, DR, BS, inv_scale);
  else
    mla_reshape_and_cache_kernel<false><<<T, 128, 0, stream>>>(
        (const uint16_t*)latent, (const uint16_t*)k_rope, cache, slot_mapping,
        R, DR, BS, inv_scale);
}

// ---- MLA: rope, latent norm and cache scatter ----------------------------------------
// Of kv [T, R + DR] the latent's RMS norm and the rotated key go to the cache, and the
// rotated part of q [T, H, DR] to rows of its own: one launch for two copies, rope, norm
// and scatter. The first block of a token has its cache row, the others 256 pieces of 8
// values of q each. Bound by latency at decode, 40 tokens x 128 heads 5 us (five
// launches of 3 to 7 before), by memory at prefill, 2,500 tokens 22 us
// or 3.7 TB/s (58 before).
// splits > 0: kv is still the fp32 parts [splits, T, R + DR] of its product over few
// rows. The first block adds them up as skinny_sum_kernel does, rounds the row to LDS
// and goes on from there, one launch less. Whole fp8 MLA layers of hidden size 7168,
// apart / so: 20 requests 241.4 / 237.2 us, 40 296.4 / 293.5, 64 302.2 / 301.4; in bf16
// 17 305.2 / 302.5, 64 370.0 / 367.9.

template <bool NEOX, bool FP8, bool PARTS>
__global__ __launch_bounds__(256) void mla_rope_and_cache_kernel(
    uint16_t* __restrict__ q_out,    // [T, H, DR]
    const uint16_t* __restrict__ q,  // [T, H, DR] by strides
    const void* __restrict__ kv,     // [T, R + DR] rows at kv_stride, or parts
    const uint16_t* __restrict__ w, void* __restrict__ cache,
    const int* __restrict__ positions, const float* __restrict__ cos_sin,
    const int64_t* __restrict__ slot_mapping, const int H, const int R,
    const int DR, const int64_t q_token, const int64_t q_head,
    const int64_t kv_stride, const int splits, const float eps) {
  __shared__ float red[16];
  extern __shared__ __attribute__((aligned(16))) uint16_t kv_row[];  // PARTS: [R + DR]
  const int t = blockIdx.x, tid = threadIdx.x;
  const int half = DR / 2;
  // 16 rotated values of src, piece `piece` of half / 8: o[0 .. 7] go to i1, the
  // others to i2
  auto rotate = [&](const uint16_t* src, int piece, float (&o)[16], int& i1,
                    int& i2) {
    const int j = piece * 8;
    const float* cs = cos_sin + (size_t)positions[t] * DR + j;
    float c[8], ss[8], x[16];
#pragma unroll
    for (int r = 0; r < 8; r += 4) {
      *reinterpret_cast<f32x4v*>(c + r) = *reinterpret_cast<const f32x4v*>(cs + r);
      *reinterpret_cast<f32x4v*>(ss + r) =
          *reinterpret_cast<const f32x4v*>(cs + half + r);
    }
    i1 = NEOX ? j : 2 * j;
    i2 = NEOX ? j + half : 2 * j + 8;
    const bf16x8 a = load_bf16x8(src + i1), b = load_bf16x8(src + i2);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      x[r] = bf16x8_get(a, r);
      x[8 + r] = bf16x8_get(b, r);
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int n1 = NEOX ? r : 2 * r, n2 = NEOX ? 8 + r : 2 * r + 1;
      o[n1] = fmaf(x[n1], c[r], -x[n2] * ss[r]);
      o[n2] = fmaf(x[n2], c[r], x[n1] * ss[r]);
    }
  };
  if (blockIdx.y > 0) {
    const int e = (blockIdx.y - 1) * 256 + tid;
    const int h = e / (half / 8), piece = e % (half / 8);
    if (h >= H) return;
    float o[16];
    int i1, i2;
    rotate(q + t * q_token + h * q_head, piece, o, i1, i2);
    uint16_t* dst = q_out + ((size_t)t * H + h) * DR;
    store_bf16x8(dst + i1, o);
    store_bf16x8(dst + i2, o + 8);
    return;
  }
  const int64_t slot = slot_mapping[t];
  if (slot < 0) return;
  const size_t row = (size_t)slot * (R + DR);
  auto put = [&](int at, const float* v) {  // as bf16, and from there fp8
    uint16_t b[8];
    store_bf16x8(b, v);
    if constexpr (FP8) {
      uint64_t o = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        o |= (uint64_t)f32_to_fp8_e4m3(bf16_bits_to_f32(b[j])) << (8 * j);
      *reinterpret_cast<uint64_t*>((uint8_t*)cache + row + at) = o;
    } else {
      *reinterpret_cast<int4*>((uint16_t*)cache + row + at) =
          *reinterpret_cast<const int4*>(b);
    }
  };
  const uint16_t* src = PARTS ? kv_row : (const uint16_t*)kv + t * kv_stride;
  if constexpr (PARTS) {
    const int N = R + DR;
    const size_t all = (size_t)gridDim.x * N;
    for (int n = tid * 4; n < N; n += 1024) {
      const float* part = (const float*)kv + (size_t)t * N + n;
      f32x4v s = {};
#pragma unroll 8
      for (int k = 0; k < splits; ++k)
        s += *reinterpret_cast<const f32x4v*>(part + k * all);
#pragma unroll
      for (int r = 0; r < 4; ++r) kv_row[n + r] = f32_to_bf16_bits(s[r]);
    }
    __syncthreads();
  }
  if (tid >= 192 && tid - 192 < half / 8) {  // the last wave, where R <= 1536 idle
    float o[16];
    int i1, i2;
    rotate(src + R, tid - 192, o, i1, i2);
    put(R + i1, o);
    put(R + i2, o + 8);
  }
  float ss = 0.f;
  for (int i = tid * 8; i < R; i += 2048) {
    const bf16x8 x = load_bf16x8(src + i);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = bf16x8_get(x, j);
      ss = fmaf(v, v, ss);
    }
  }
  ss = block_reduce_sum(ss, red);
  const float rstd = rsqrtf(ss / R + eps);
  for (int i = tid * 8; i < R; i += 2048) {
    const bf16x8 x = load_bf16x8(src + i), g = load_bf16x8(w + i);
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = bf16x8_get(x, j) * rstd * bf16x8_get(g, j);
    put(i, v);
  }
}

// splits 0: kv is bf16 rows
extern "C" void launch_mla_rope_and_cache(
    void* q_out, const void* q, const void* kv, const void* w, void* cache,
    const int* positions, const float* cos_sin, const int64_t* slot_mapping, int T,
    int H, int R, int DR, int64_t q_token, int64_t q_head, int64_t kv_stride,
    int splits, float eps, bool neox, bool fp8, hipStream_t stream) {
  const dim3 grid(T, 1 + ceil_div(H * (DR / 16), 256));
  auto run = [&](auto kernel, int lds) {
    kernel<<<grid, 256, lds, stream>>>(
        (uint16_t*)q_out, (const uint16_t*)q, kv, (const uint16_t*)w, cache, positions,
        cos_sin, slot_mapping, H, R, DR, q_token, q_head, kv_stride, splits, eps);
  };
  auto by = [&](auto n, auto f) {
    constexpr bool N = decltype(n)::value, F = decltype(f)::value;
    if (splits > 0) run(mla_rope_and_cache_kernel<N, F, true>, (R + DR) * 2);
    else run(mla_rope_and_cache_kernel<N, F, false>, 0);
  };
  auto of = [&](auto n) {
    if (fp8) by(n, std::true_type{});
    else by(n, std::false_type{});
  };
  if (neox) of(std::true_type{});
  else of(std::false_type{});
}

// ---- activations ----------------------------------------------------------------------
// x: [T, 2I] (gate | up) -> out: [T, I];  grid-stride, vectorized.

// MAX: part[block] is the largest magnitude among the block's results, as bits, for a
// conversion to fp8 without a pass of its own to find it: 40 rows of 18432 8.0 to 6.7 us
// with the conversion, one row 6.6 to 5.3
template <bool GELU, bool MAX>
__global__ void act_and_mul_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
    uint32_t* __restrict__ part, const int64_t T, const int I) {
  uint32_t top = 0;
  const int64_t total = T * (I / 8);
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = idx / (I / 8);
    const int i = (idx % (I / 8)) * 8;
    bf16x8 g = load_bf16x8(x + t * 2 * I + i);
    bf16x8 u = load_bf16x8(x + t * 2 * I + I + i);
    float vals[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float gv = bf16x8_get(g, j);
      const float uv = bf16x8_get(u, j);
      float a;
      if (GELU) {  // tanh approximation
        const float c = 0.7978845608028654f;
        a = 0.5f * gv * (1.f + tanhf(c * (gv + 0.044715f * gv * gv * gv)));
      } else {  // silu
        a = gv / (1.f + __expf(-gv));
      }
      vals[j] = a * uv;
    }
    bf16x8 o;
    store_bf16x8(&o, vals);
    *reinterpret_cast<int4*>(out + t * I + i) = o.raw;
    if (MAX) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        top = max(top, __float_as_uint(bf16x8_get(o, j)) & 0x7fffffffu);
    }
  }
  if (MAX) {
    __shared__ uint32_t tops[4];  // 256 threads
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
      top = max(top, (uint32_t)__shfl_xor((int)top, o, WAVE_SIZE));
    if ((threadIdx.x & 63) == 0) tops[threadIdx.x >> 6] = top;
    __syncthreads();
    if (threadIdx.x == 0)
      part[blockIdx.x] = max(max(tops[0], tops[1]), max(tops[2], tops[3]));
  }
}

// parts of silu_and_mul's results whose largest magnitudes launch_silu_and_mul_max gives
extern "C" int silu_and_mul_parts(int64_t T, int I) {
  return clamp_int((T * (I / 8) + 255) / 256, 1, 1024);
}
extern "C" void launch_silu_and_mul_max(void* out, uint32_t* part, const void* x,
                                        int64_t T, int I, hipStream_t stream) {
  act_and_mul_kernel<false, true><<<silu_and_mul_parts(T, I), 256, 0, stream>>>(
      (uint16_t*)out, (const uint16_t*)x, part, T, I);
}

extern "C" void launch_act_and_mul(
    void* out, const void* x, int64_t T, int I, bool gelu, hipStream_t stream) {
  long long total = (long long)T * (I / 8);
  int blocks = clamp_int((total + 255) / 256, 1, 2048);
  if (gelu)
    act_and_mul_kernel<true, false><<<blocks, 256, 0, stream>>>(
        (uint16_t*)out, (const uint16_t*)x, nullptr, T, I);
  else
    act_and_mul_kernel<false, false><<<blocks, 256, 0, stream>>>(
        (uint16_t*)out, (const uint16_t*)x, nullptr, T, I);
}
