// Routed experts for gfx950: device-side routing, two grouped GEMMs, a combine.
//
//   moe_route      counts the choices of every expert, sorts them (perm: sorted
//                  place -> flat choice t * k + j) and lists the tiles of TM
//                  rows; one workgroup, no host involvement
//   moe_gemm<GATE> h = act(x[gather] . W_gu[e]^T): gate and up columns meet in
//                  the same lane, the activation is applied in registers
//   moe_gemm       y[choice] = w * (h . W_down[e]^T), fp32
//   moe_combine    out[t] = sum of its choices' y, in the order of the choices
// With in_w the routing weight multiplies the expert's INPUT instead: the
// gate/up accumulators are scaled by it (both projections are linear).
// fp8: W8A8, weights e4m3 with a scale per output row, activations quantised a
// row (x before the first product, h before the second).
//
// W_gu is [E, 2I, H], W_down [E, H, I]. Choices of an expert outside [0, E) (the
// experts of another rank) are left out. Grids are upper bounds (blocks past
// the live tiles exit), so a captured step replays with any routing.

#include "common.h"

#include <type_traits>

#define MOE_BKB 128    // bytes of the contraction a stage

typedef float f32x16v __attribute__((ext_vector_type(16)));
typedef int i32x4v __attribute__((ext_vector_type(4)));
typedef int i32x8v __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2n __attribute__((ext_vector_type(2)));

namespace {

DEVINL uint32_t pack_bf16(float a, float b) {
  bf16x2n p;
  p[0] = (__bf16)a;
  p[1] = (__bf16)b;
  return __builtin_bit_cast(uint32_t, p);
}

DEVINL void copy16_to_lds(const void* src, void* dst) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)src,
      (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

}  // namespace

// ---- routing ------------------------------------------------------------------
// perm [n], tiles [max_tiles] as (expert, first row, end of the expert's rows,
// -), n_tiles [1]. A decode step has a few hundred choices: one workgroup and
// one launch do it in 5 us. LDS counters bound it, 60 cycles an atomic of a
// wave: 65,536 choices took one workgroup 52 us, so parts of ROUTE_PART choices
// are counted first (moe_count), and each then places its own behind the
// parts before it.

#define ROUTE_THREADS 1024
#define ROUTE_PART 4096
#define ROUTE_LDS 8192  // experts whose counters fit the LDS

// The counters of more experts lie in memory and belong to one workgroup, which
// goes by atomic operations only: plain ones may meet its own cache.
template <bool LDS>
DEVINL int get_count(const int* p) {
  return LDS ? *p
             : __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool LDS>
DEVINL void set_count(int* p, int v) {
  if (LDS) *p = v;
  else __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool LDS>
DEVINL void route_sync() {
  if (!LDS) __threadfence();
  __syncthreads();
}

// cnt[e] += this part's choices of expert e
DEVINL void count_choices(int* cnt, const int64_t* ids, int begin, int end,
                          int E) {
  // ids are fetched four ahead of the counters, which would wait for each
  constexpr int AHEAD = ROUTE_PART / ROUTE_THREADS;
  for (int i0 = begin + threadIdx.x; i0 < end; i0 += ROUTE_PART) {
    int64_t e[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int i = i0 + u * ROUTE_THREADS;
      e[u] = i < end ? ids[i] : -1;
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (e[u] >= 0 && e[u] < E) atomicAdd(&cnt[e[u]], 1);
  }
}

__global__ __launch_bounds__(ROUTE_THREADS) void moe_count_kernel(
    int* __restrict__ counts,  // [parts, E]
    const int64_t* __restrict__ ids, const int n, const int E) {
  extern __shared__ int lds[];
  for (int e = threadIdx.x; e < E; e += ROUTE_THREADS) lds[e] = 0;
  __syncthreads();
  const int begin = blockIdx.x * ROUTE_PART;
  count_choices(lds, ids, begin, min(n, begin + ROUTE_PART), E);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += ROUTE_THREADS)
    counts[(size_t)blockIdx.x * E + e] = lds[e];
}

template <bool LDS>
__global__ __launch_bounds__(ROUTE_THREADS) void moe_route_kernel(
    int* __restrict__ perm, int4* __restrict__ tiles, int* __restrict__ n_tiles,
    int* __restrict__ counts, const int64_t* __restrict__ ids,
    const int n, const int E, const int tm) {
  extern __shared__ int lds[];
  int* cur = LDS ? lds : counts;  // counters, then every expert's next place
  __shared__ int wave_rows[16], wave_tiles[16];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6;
  const int parts = gridDim.x;
  const int begin = parts > 1 ? blockIdx.x * ROUTE_PART : 0;
  const int end = parts > 1 ? min(n, begin + ROUTE_PART) : n;
  if (parts == 1) {
    for (int e = tid; e < E; e += ROUTE_THREADS) set_count<LDS>(cur + e, 0);
    route_sync<LDS>();
    count_choices(cur, ids, begin, end, E);
    route_sync<LDS>();
  }
  // exclusive sums of rows and tiles over the experts, 1024 at a time
  int rows0 = 0, tiles0 = 0;
  for (int e0 = 0; e0 < E; e0 += ROUTE_THREADS) {
    const int e = e0 + tid;
    int c = 0, before = 0;
    if (e < E) {
      if (parts == 1) {
        c = get_count<LDS>(cur + e);
      } else {
        for (int q = 0; q < parts; ++q) {
          const int v = counts[(size_t)q * E + e];
          c += v;
          before += q < (int)blockIdx.x ? v : 0;
        }
      }
    }
    const int t = (c + tm - 1) / tm;
    int rs = c, ts = t;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int r2 = __shfl_up(rs, o, WAVE_SIZE);
      const int t2 = __shfl_up(ts, o, WAVE_SIZE);
      if (lane >= o) {
        rs += r2;
        ts += t2;
      }
    }
    if (lane == 63) {
      wave_rows[wid] = rs;
      wave_tiles[wid] = ts;
    }
    __syncthreads();
    int rb = rows0, tb = tiles0, rsum = 0, tsum = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      if (w < wid) {
        rb += wave_rows[w];
        tb += wave_tiles[w];
      }
      rsum += wave_rows[w];
      tsum += wave_tiles[w];
    }
    if (e < E) {
      const int r0 = rb + rs - c;
      int at = tb + ts - t;
      set_count<LDS>(cur + e, r0 + before);
      if (blockIdx.x == 0)
        for (int r = r0; r < r0 + c; r += tm)
          tiles[at++] = make_int4(e, r, r0 + c, 0);
    }
    rows0 += rsum;
    tiles0 += tsum;
    route_sync<LDS>();
  }
  if (tid == 0 && blockIdx.x == 0) *n_tiles = tiles0;
  constexpr int AHEAD = ROUTE_PART / ROUTE_THREADS;
  for (int i0 = begin + tid; i0 < end; i0 += ROUTE_PART) {
    int64_t e[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int i = i0 + u * ROUTE_THREADS;
      e[u] = i < end ? ids[i] : -1;
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (e[u] >= 0 && e[u] < E)
        perm[atomicAdd(&cur[e[u]], 1)] = i0 + u * ROUTE_THREADS;
  }
}

// ---- grouped GEMM ----------------------------------------------------------------
// A workgroup takes one tile of TM rows of one expert and TN of its weight
// rows: D[feature x row] = W . A^T on 32x32 matrix instructions, so that a lane
// ends with four neighbouring features of one row. Both operands go global ->
// LDS directly (16 bytes a lane, STAGES - 1 stages of 128 bytes of every row in
// flight), 16-byte chunks XOR-swizzled by row so that 16 rows of one chunk
// column lie in 16 bank groups.
//   TM 32, 64: the weights' stream is the work. 4 waves x 32 weight rows.
//   TM 128:    matrix products, 256 weight rows: 4 x 2 waves of 64 x 64.
// GATE: of 32 weight rows of a wave 16 are gate and 16 the up rows of the same
// columns; the accumulator's upper registers are the lower ones' partners.
// What bounds it: few rows, the weights' stream: 256 fp8 experts of 7168 x 2048,
// 200 tokens x 8 choices, gate/up 0.99 ms and down 0.55 ms = 6.2 TB/s of the
// experts touched (2.44 and 1.06 ms with fragments loaded straight to
// registers). Many rows, the address unit: it moves 64 bytes a cycle and CU, so
// a 128 x 256 tile takes 768 of its cycles for 1024 of the matrix cores (128 x
// 128: 512 for 512), and copies asked for in one burst hold their wave up: they
// are spread over the products. 128 bf16 experts of 2048 x 768, 8192 tokens x 8:
// gate/up 585 us = 705 TFLOP/s, down 450 us in two slabs (2247 and 1530 us before).

struct MoeArgs {
  const uint8_t* w;        // [E, w_rows, kb] bytes
  const float* w_scale;    // [E, w_rows] (fp8)
  const uint8_t* a;        // rows of kb bytes: x [T] or h [n]
  const float* a_scale;    // per row of a (fp8)
  const int* perm;
  const int4* tiles;
  const int* n_tiles;
  const float* choice_w;   // [T, k] routing weights
  const uint16_t* bias;    // [E, 2I] or null (GATE)
  void* out;               // GATE: h [n, N] bf16; else y [T * k, cols] fp32
  int topk, N, kb, nb;     // N output features, kb bytes a row, nb column blocks
  int first, cols;         // the features of this launch: all (GATE), or a slab
  int in_w, gelu;
  float limit;             // > 0: clamped activation
};

template <bool FP8, int TN, int TM, bool GATE, int STAGES>
__global__ __launch_bounds__(2 * TN, 2) void moe_gemm_kernel(const MoeArgs p) {
  constexpr int WN = TM == 128 ? 2 : 1;  // 32-row weight tiles a wave
  constexpr int WM = TM == 32 ? 1 : 2;   // 32-row activation tiles a wave
  constexpr int PASS = TN / 4;            // rows the threads copy at once
  constexpr int APASS = TM / PASS;
  constexpr int LOADS = 4 + APASS;        // copies a thread and stage
  constexpr int BUF = (TN + TM) * MOE_BKB;
  __shared__ __attribute__((aligned(16))) uint8_t S0[BUF];
  __shared__ __attribute__((aligned(16))) uint8_t S1[BUF];
  __shared__ __attribute__((aligned(16))) uint8_t S2[BUF];
  __shared__ __attribute__((aligned(16))) uint8_t S3[STAGES > 3 ? BUF : 16];

  // Blocks go round-robin to the 8 XCDs. Each XCD takes a contiguous eighth of
  // the (tile, column block) list, so that the blocks of an expert share one
  // L2: its weights and rows are read from memory once.
  const int total = *p.n_tiles * p.nb;
  const int chunk = (total + 7) >> 3;
  const int slot = blockIdx.x >> 3;
  const int idx = (blockIdx.x & 7) * chunk + slot;
  if (slot >= chunk || idx >= total) return;
  const int4 tile = p.tiles[idx / p.nb];
  const int e = __builtin_amdgcn_readfirstlane(tile.x);
  const int row0 = __builtin_amdgcn_readfirstlane(tile.y);
  const int rows_end = __builtin_amdgcn_readfirstlane(tile.z);
  const int n0 = p.first + (idx % p.nb) * (GATE ? TN / 2 : TN);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  const int l31 = lane & 31;

  // ---- what a thread copies: one chunk of rows tid / 8 + PASS i --------------------
  const int src = (tid & 7) ^ ((tid >> 4) & 7);
  const uint8_t* wp[4];
  const uint8_t* ap[APASS];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = i * PASS + (tid >> 3);
    int row;  // rows past the last feature are read twice and never stored
    if (GATE)
      row = ((r >> 4) & 1) * p.N + min(n0 + (r >> 5) * 16 + (r & 15), p.N - 1);
    else
      row = min(n0 + r, p.N - 1);
    wp[i] = p.w + ((size_t)e * (GATE ? 2 * p.N : p.N) + row) * p.kb;
  }
#pragma unroll
  for (int i = 0; i < APASS; ++i) {
    const int r = min(row0 + i * PASS + (tid >> 3), rows_end - 1);
    ap[i] = p.a + (size_t)(GATE ? p.perm[r] / p.topk : r) * p.kb;
  }
  // copy i of a stage: 4 passes over the weight rows, then the activation rows
  auto copy = [&](int i, int off, uint8_t* S) {
    if (i < 4)
      copy16_to_lds(wp[i] + off, S + (i * PASS + wid * 8) * MOE_BKB);
    else
      copy16_to_lds(ap[i - 4] + off,
                    S + (TN + (i - 4) * PASS + wid * 8) * MOE_BKB);
  };
  auto offset = [&](int kt) {
    return min(kt * MOE_BKB + src * 16, p.kb - 16);
  };
  auto issue = [&](int kt, uint8_t* S) {
    const int off = offset(kt);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) copy(i, off, S);
  };

  // waves: TM 128: TN / 64 x 2 of 64 x 64; else TN / 32 x 1 of 32 x TM
  const int wb = TM == 128 ? (wid & (TN / 64 - 1)) * 64 : wid * 32;
  const int ab = TM == 128 ? wid / (TN / 64) * 64 : 0;
  const int swz_l = (l31 >> 1) & 7;
  using frag_t = std::conditional_t<FP8, i32x8v, bf16x8v>;
  f32x16v acc[WN][WM] = {};

  // FULL: 128 bytes of the contraction; else what is left of it (32 k bytes).
  auto stage = [&](const uint8_t* S, int left, auto full, auto&& between) {
    constexpr bool FULL = decltype(full)::value;
    constexpr int KS = FP8 ? 2 : 4;
    const uint8_t* Wl = S + (wb + l31) * MOE_BKB;
    const uint8_t* Al = S + (TN + ab + l31) * MOE_BKB;
    frag_t a[2][WN], b[2][WM];
    auto fetch = [&](int ks) {
#pragma unroll
      for (int i = 0; i < WN + WM; ++i) {
        const uint8_t* r = i < WN ? Wl + i * 32 * MOE_BKB
                                  : Al + (i - WN) * 32 * MOE_BKB;
        frag_t& f = i < WN ? a[ks & 1][i] : b[ks & 1][i - WN];
        if constexpr (FP8) {
          const int c0 = ((4 * ks + 2 * half) ^ swz_l) * 16;
          const int c1 = ((4 * ks + 2 * half + 1) ^ swz_l) * 16;
          f = __builtin_shufflevector(*(const i32x4v*)(r + c0),
                                      *(const i32x4v*)(r + c1), 0, 1, 2, 3, 4,
                                      5, 6, 7);
          // of a last step of 32 the upper half of the lanes has nothing, and
          // of a step behind the end no lane has
          if (!FULL && left - ks * 64 < (half ? 64 : 1)) f = 0;
        } else {
          f = *(const bf16x8v*)(r + ((2 * ks + half) ^ swz_l) * 16);
          if (!FULL && ks * 32 >= left) f = 0;
        }
      }
    };
    // lgkmcnt(0) before the next step's operands are asked for: this step's
    // products need no further wait and run while those are under way
    auto landed = [] {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_sched_barrier(0);
    };
    fetch(0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      landed();
      if (ks + 1 < KS) fetch(ks + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < WN; ++i)
#pragma unroll
        for (int j = 0; j < WM; ++j) {
          if constexpr (FP8)
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                a[ks & 1][i], b[ks & 1][j], acc[i][j], 0, 0, 0, 0x7f7f7f7f, 0,
                0x7f7f7f7f);
          else
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                a[ks & 1][i], b[ks & 1][j], acc[i][j], 0, 0, 0);
          between((ks * WN + i) * WM + j);
        }
    }
  };

  // One barrier a stage: behind it stage kt is in LDS for every wave, and the
  // buffer that stage kt + STAGES - 1 goes to has been left by every wave. Past
  // the end the copies go on, of one cached chunk a row, so that the number of
  // copies in flight is the same for every stage and the wait a constant.
  auto turn = [&](int kt, uint8_t* S, uint8_t* Sn) {
    constexpr int V = (STAGES - 2) * LOADS;  // copies of the later stages
    // a fence would wait for every copy: vmcnt(V), lgkmcnt(0) by hand, and no
    // LDS access moves over the barrier
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070 | (V & 15) | ((V >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // the copies are spread over the products: a wave that asks for all of
    // them at once waits for the address unit, which takes 64 bytes a cycle
    const int off = offset(kt + STAGES - 1);
    constexpr int PRODUCTS = (FP8 ? 2 : 4) * WN * WM;
    stage(S, MOE_BKB, std::true_type{}, [&](int m) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i)
        if (m == i * PRODUCTS / LOADS) {
          __builtin_amdgcn_sched_barrier(0);
          copy(i, off, Sn);
          __builtin_amdgcn_sched_barrier(0);
        }
    });
  };
  const int nk = p.kb / MOE_BKB;  // full stages
  issue(0, S0);
  issue(1, S1);
  if constexpr (STAGES > 3) issue(2, S2);
  for (int kt = 0; kt < nk;) {
    turn(kt, S0, STAGES == 3 ? S2 : S3);
    if (++kt >= nk) break;
    turn(kt, S1, S0);
    if (++kt >= nk) break;
    turn(kt, S2, S1);
    if (++kt >= nk) break;
    if constexpr (STAGES > 3) {
      turn(kt, S3, S2);
      if (++kt >= nk) break;
    }
  }
  // the last copies: no more may land in LDS once the workgroup has ended
  __builtin_amdgcn_s_waitcnt(0x0f70);
  if (p.kb % MOE_BKB) {
    __syncthreads();
    const int at = nk % STAGES;
    stage(at == 0 ? S0 : at == 1 ? S1 : at == 2 ? S2 : S3, p.kb % MOE_BKB,
          std::false_type{}, [](int) {});
  }

  // ---- results: column = row of the tile, registers = features --------------------
#pragma unroll
  for (int j = 0; j < WM; ++j) {
    const int r = row0 + ab + j * 32 + l31;
    if (r >= rows_end) continue;
    const int choice = p.perm[r];
    const float w = p.choice_w[choice];
    const float sa = FP8 ? p.a_scale[GATE ? choice / p.topk : r] : 1.f;
#pragma unroll
    for (int i = 0; i < WN; ++i) {
      if (GATE) {
        uint16_t* h = (uint16_t*)p.out + (size_t)r * p.N;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int f = n0 + (wb >> 1) + i * 16 + 8 * q + 4 * half;
          if (f >= p.N) continue;
          float v[4];
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            float g = acc[i][j][4 * q + s], u = acc[i][j][8 + 4 * q + s];
            if (FP8) {
              const float* ws = p.w_scale + (size_t)e * 2 * p.N + f + s;
              g *= sa * ws[0];
              u *= sa * ws[p.N];
            }
            if (p.in_w) {
              g *= w;
              u *= w;
            }
            if (p.bias != nullptr) {
              const uint16_t* b = p.bias + (size_t)e * 2 * p.N + f + s;
              g += bf16_bits_to_f32(b[0]);
              u += bf16_bits_to_f32(b[p.N]);
            }
            if (p.limit > 0.f) {  // gpt-oss clamped act
              g = fminf(g, p.limit);
              u = fminf(fmaxf(u, -p.limit), p.limit);
              v[s] = (u + 1.f) * (g / (1.f + __expf(-g * 1.702f)));
            } else if (p.gelu) {
              const float c = 0.7978845608028654f;
              v[s] =
                  0.5f * g * (1.f + tanhf(c * (g + 0.044715f * g * g * g))) * u;
            } else {
              v[s] = g / (1.f + __expf(-g)) * u;
            }
          }
          uint2 o;
          o.x = pack_bf16(v[0], v[1]);
          o.y = pack_bf16(v[2], v[3]);
          *reinterpret_cast<uint2*>(h + f) = o;
        }
      } else {
        float* y = (float*)p.out + (size_t)choice * p.cols - p.first;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int f = n0 + wb + i * 32 + 8 * q + 4 * half;
          if (f >= p.first + p.cols) continue;
          f32x4v o;
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            float c = p.in_w ? 1.f : w;
            if (FP8) c *= sa * p.w_scale[(size_t)e * p.N + f + s];
            o[s] = acc[i][j][4 * q + s] * c;
          }
          *reinterpret_cast<f32x4v*>(y + f) = o;
        }
      }
    }
  }
}

// ---- combine --------------------------------------------------------------------
// out[t] = sum over its choices, of the features from first on; four a thread.

__global__ __launch_bounds__(256) void moe_combine_kernel(
    float* __restrict__ out, const float* __restrict__ y,
    const int64_t* __restrict__ ids, const int T, const int k, const int E,
    const int H, const int first, const int cols) {
  const int t = blockIdx.x;
  for (int c = (blockIdx.y * 256 + threadIdx.x) * 4; c < cols;
       c += gridDim.y * 1024) {
    f32x4v s = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < k; ++j) {
      const int64_t e = ids[(size_t)t * k + j];
      if (e >= 0 && e < E)
        s += *reinterpret_cast<const f32x4v*>(y + ((size_t)t * k + j) * cols + c);
    }
    *reinterpret_cast<f32x4v*>(out + (size_t)t * H + first + c) = s;
  }
}

// ---- activations to fp8 (OCP e4m3), one scale a row --------------------------------

#define FP8_MAX 448.f

__global__ __launch_bounds__(256) void quantize_fp8_rows_kernel(
    uint8_t* __restrict__ out,      // [R, C]
    float* __restrict__ scales,     // [R] dequant scale (amax/448)
    const uint16_t* __restrict__ x, // [R, C] bf16
    const int C) {
  const int row = blockIdx.x;
  const uint16_t* xr = x + (size_t)row * C;
  uint8_t* orow = out + (size_t)row * C;
  float amax = 1e-8f;
  for (int c = threadIdx.x * 8; c < C; c += blockDim.x * 8) {
    bf16x8 v = load_bf16x8(xr + c);
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(bf16x8_get(v, i)));
  }
  __shared__ float lds[8];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  amax = wave_reduce_max(amax);
  if (lane == 0) lds[wid] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(lds[0], lds[1]), fmaxf(lds[2], lds[3]));
  if (threadIdx.x == 0) scales[row] = amax / FP8_MAX;
  const float inv = FP8_MAX / amax;
  for (int c = threadIdx.x * 8; c < C; c += blockDim.x * 8) {
    bf16x8 v = load_bf16x8(xr + c);
    uint64_t qv = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      qv |= (uint64_t)f32_to_fp8_e4m3(bf16x8_get(v, i) * inv) << (8 * i);
    *reinterpret_cast<uint64_t*>(orow + c) = qv;
  }
}

extern "C" void launch_quantize_fp8_rows(
    void* out, float* scales, const void* x, int R, int C,
    hipStream_t stream) {
  quantize_fp8_rows_kernel<<<R, 256, 0, stream>>>(
      (uint8_t*)out, scales, (const uint16_t*)x, C);
}

// ---- the two products of a layer -----------------------------------------------

template <bool FP8, int TN, int TM, int STAGES>
static void launch_gemm(bool gate, MoeArgs& p, int max_tiles,
                        hipStream_t stream) {
  p.nb = ceil_div(p.cols, gate ? TN / 2 : TN);
  const int blocks = (max_tiles * p.nb + 7) / 8 * 8;
  if (gate)
    moe_gemm_kernel<FP8, TN, TM, true, STAGES>
        <<<blocks, 2 * TN, 0, stream>>>(p);
  else
    moe_gemm_kernel<FP8, TN, TM, false, STAGES>
        <<<blocks, 2 * TN, 0, stream>>>(p);
}

template <bool FP8>
static void launch_gemm_tm(int tm, bool gate, MoeArgs& p, int max_tiles,
                           hipStream_t stream) {
  if (tm == 32)
    launch_gemm<FP8, 128, 32, 4>(gate, p, max_tiles, stream);
  else if (tm == 64)
    launch_gemm<FP8, 128, 64, 3>(gate, p, max_tiles, stream);
  else
    launch_gemm<FP8, 256, 128, 3>(gate, p, max_tiles, stream);
}

// Rows a tile, by the mean number of choices an expert. Measured (us, tiles of
// 32 / 64 / 128 rows): bf16 128 experts of 2048 x 768, mean 6: 182 / 189 / 230,
// 25: 251 / 246 / 247, 43: 326 / 284 / 311, 62: 390 / 338 / 319, 512: 1855 /
// 1378 / 1089; 32 experts of 2048 x 1024, mean 25: 106 / 122 / 151, 62: 148 /
// 123 / 156, 250: 353 / 252 / 223; fp8 256 experts of 7168 x 2048, mean 6: 1334 /
// 1296 / 1360, 21: 2167 / 1926 / 1989, 46: 3178 / 2503 / 2306. Below, the
// weights' stream is the work and few rows cost nothing; 128 rows pay earlier
// where there are blocks enough for the chip (8 a CU).
extern "C" int moe_tile_rows(int n, int E, int I, bool fp8) {
  const int mean = n / (E > 0 ? E : 1);
  if (mean <= (fp8 ? 12 : 24)) return 32;
  const int64_t blocks = ((int64_t)n / 128 + E / 2) * ceil_div(I, 128);
  return mean > 96 || (mean > 40 && blocks >= 2048) ? 128 : 64;
}

extern "C" int moe_max_tiles(int n, int E, int tm) {
  return n / tm + (n < E ? n : E);
}

// Output features of a down product and combine: y takes at most MOE_Y_BYTES (of
// 256 features, a tile's width, at least), however many tokens a step brings. 65,536
// choices of 2048 features, a whole call: one slab of 537 MB 1.033 ms, two of 256
// MB at most 1.030.
#define MOE_Y_BYTES (256ll << 20)
extern "C" int moe_down_cols(int n, int H) {
  const int64_t cols = MOE_Y_BYTES / (4ll * n) & ~255ll;
  return cols >= H ? H : cols < 256 ? (H < 256 ? H : 256) : (int)cols;
}

// ints of scratch that routing n choices takes besides perm and tiles
static int route_parts(int n, int E) {
  return n > 2 * ROUTE_PART && E <= ROUTE_LDS ? ceil_div(n, ROUTE_PART) : 1;
}
extern "C" int64_t moe_route_scratch(int n, int E) {
  const int parts = route_parts(n, E);
  return parts > 1 || E > ROUTE_LDS ? (int64_t)parts * E : 0;
}

extern "C" void launch_moe_route(int* perm, void* tiles, int* n_tiles,
                                 int* counts, const int64_t* ids, int n, int E,
                                 int tm, hipStream_t stream) {
  const int parts = route_parts(n, E);
  if (E > ROUTE_LDS) {
    moe_route_kernel<false><<<1, ROUTE_THREADS, 0, stream>>>(
        perm, (int4*)tiles, n_tiles, counts, ids, n, E, tm);
    return;
  }
  if (parts > 1)
    moe_count_kernel<<<parts, ROUTE_THREADS, E * sizeof(int), stream>>>(
        counts, ids, n, E);
  moe_route_kernel<true><<<parts, ROUTE_THREADS, E * sizeof(int), stream>>>(
      perm, (int4*)tiles, n_tiles, counts, ids, n, E, tm);
}

extern "C" void launch_moe_gate_up(
    void* h, const void* x, const float* x_scale, const void* w_gu,
    const float* w_scale, const int* perm, const void* tiles,
    const int* n_tiles, const float* choice_w, const void* bias, int topk,
    int H, int I, int max_tiles, int tm, bool fp8, bool in_w, bool gelu,
    float limit, hipStream_t stream) {
  MoeArgs p{(const uint8_t*)w_gu, w_scale, (const uint8_t*)x, x_scale, perm,
            (const int4*)tiles, n_tiles, choice_w, (const uint16_t*)bias, h,
            topk, I, fp8 ? H : 2 * H, 0, 0, I, in_w, gelu,
            limit};
  if (fp8)
    launch_gemm_tm<true>(tm, true, p, max_tiles, stream);
  else
    launch_gemm_tm<false>(tm, true, p, max_tiles, stream);
}

extern "C" void launch_moe_down(
    float* y, const void* h, const float* h_scale, const void* w_down,
    const float* w_scale, const int* perm, const void* tiles,
    const int* n_tiles, const float* choice_w, int topk, int H, int I,
    int first, int cols, int max_tiles, int tm, bool fp8, bool in_w,
    hipStream_t stream) {
  MoeArgs p{(const uint8_t*)w_down, w_scale, (const uint8_t*)h, h_scale, perm,
            (const int4*)tiles, n_tiles, choice_w, nullptr, y, topk, H,
            fp8 ? I : 2 * I, 0, first, cols, in_w, 0, 0.f};
  if (fp8)
    launch_gemm_tm<true>(tm, false, p, max_tiles, stream);
  else
    launch_gemm_tm<false>(tm, false, p, max_tiles, stream);
}

extern "C" void launch_moe_combine(float* out, const float* y,
                                   const int64_t* ids, int T, int k, int E,
                                   int H, int first, int cols,
                                   hipStream_t stream) {
  dim3 grid(T, T < 256 ? ceil_div(cols, 1024) : 1, 1);
  moe_combine_kernel<<<grid, 256, 0, stream>>>(out, y, ids, T, k, E, H, first,
                                               cols);
}
