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

#include <type_traits>

#include "moe_common.h"

#define MOE_BKB 128    // bytes of the contraction a stage
#define MOE_UNIT (256 * MOE_BKB)

typedef float f32x16v __attribute__((ext_vector_type(16)));
typedef unsigned long long u64;

// ---- activations to fp8 (OCP e4m3), one scale a row --------------------------------

#define FP8_MAX 448.f

// Row `row` by 256 threads, tid of them; lds: four floats of theirs. The whole
// workgroup calls it, on: whether there is such a row.
DEVINL void quantize_row(uint8_t* out, float* scales, const uint16_t* x, int row,
                         int C, int tid, float* lds, bool on) {
  const uint16_t* xr = x + (size_t)row * C;
  uint8_t* orow = out + (size_t)row * C;
  const int end = on ? C : 0;
  float amax = 1e-8f;
  for (int c = tid * 8; c < end; c += 2048) {
    bf16x8 v = load_bf16x8(xr + c);
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(bf16x8_get(v, i)));
  }
  amax = wave_reduce_max(amax);
  if ((tid & 63) == 0) lds[tid >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(lds[0], lds[1]), fmaxf(lds[2], lds[3]));
  if (on && tid == 0) scales[row] = amax / FP8_MAX;
  const float inv = FP8_MAX / amax;
  for (int c = tid * 8; c < end; c += 2048) {
    bf16x8 v = load_bf16x8(xr + c);
    uint64_t qv = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      qv |= (uint64_t)f32_to_fp8_e4m3(bf16x8_get(v, i) * inv) << (8 * i);
    *reinterpret_cast<uint64_t*>(orow + c) = qv;
  }
}

__global__ __launch_bounds__(256) void quantize_fp8_rows_kernel(
    uint8_t* __restrict__ out,      // [R, C]
    float* __restrict__ scales,     // [R] dequant scale (amax/448)
    const uint16_t* __restrict__ x, // [R, C] bf16
    const int C) {
  __shared__ float lds[4];
  quantize_row(out, scales, x, blockIdx.x, C, threadIdx.x, lds, true);
}

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

// Rows that are quantised for the experts, four a workgroup behind those that route:
// neither needs the other, and a decode step's launch costs more than either. us of a
// call, a launch each / in one: 16 experts of 1024 x 512, 120 tokens 26.0 / 23.6, 849
// tokens 37.2 / 34.2; 32 of 2048 x 1024, 71 tokens 45.3 / 42.9, 294 65.5 / 63.0; 128 of
// 2048 x 768, 6,000 tokens 487 / 485; 256 of 7168 x 2048, 10 tokens 382 / 380.
struct QuantizeRows {
  uint8_t* out;        // [T, C], null: none
  float* scales;       // [T]
  const uint16_t* x;   // [T, C]
  int T, C;
};

template <bool LDS>
__global__ __launch_bounds__(ROUTE_THREADS) void moe_route_kernel(
    int* __restrict__ perm, int4* __restrict__ tiles, int* __restrict__ n_tiles,
    int* __restrict__ counts, const int64_t* __restrict__ ids,
    const int n, const int E, const int tm, const int parts, const QuantizeRows rows) {
  extern __shared__ int lds[];
  if ((int)blockIdx.x >= parts) {
    __shared__ float largest[ROUTE_THREADS / 64];
    const int grp = threadIdx.x >> 8;
    const int row = ((int)blockIdx.x - parts) * (ROUTE_THREADS / 256) + grp;
    quantize_row(rows.out, rows.scales, rows.x, row, rows.C, threadIdx.x & 255,
                 largest + grp * 4, row < rows.T);
    return;
  }
  int* cur = LDS ? lds : counts;  // counters, then every expert's next place
  __shared__ int wave_rows[16], wave_tiles[16];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6;
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
// A workgroup takes one tile of TM rows of one expert and 128 of its weight
// rows: D[feature x row] = W . A^T on 32x32 matrix instructions, so that a lane
// ends with four neighbouring features of one row. Both operands go global ->
// LDS directly (16 bytes a lane, STAGES - 1 stages of 128 bytes of every row in
// flight), 16-byte chunks XOR-swizzled by row so that 16 rows of one chunk
// column lie in 16 bank groups.
// TM 32 or 64: the weights' stream is the work. 4 waves x 32 weight rows.
// GATE: of 32 weight rows of a wave 16 are gate and 16 the up rows of the same
// columns; the accumulator's upper registers are the lower ones' partners.
// What bounds it: the weights' stream. 128 bf16 experts of 2048 x 768, 24 tokens x 8
// choices: a whole call 123 us, 126 where the compiler waited for every copy in flight
// once in STAGES stages (see copy16).

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

// ---- results: column = row of the tile, registers = features ----------------------
// A wave's 32 WN weight rows from wb on.
template <bool FP8, bool GATE, int WN, int WM>
DEVINL void store_results(const MoeArgs& p, const f32x16v (&acc)[WN][WM],
                          const int e, const int row0, const int rows_end,
                          const int n0, const int wb) {
  const int half = (threadIdx.x >> 5) & 1, l31 = threadIdx.x & 31;
#pragma unroll
  for (int j = 0; j < WM; ++j) {
    const int r = row0 + j * 32 + l31;
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

template <bool FP8, int TM, bool GATE, int STAGES>
__global__ __launch_bounds__(256, 2) void moe_gemm_kernel(const MoeArgs p) {
  constexpr int TN = 128;
  constexpr int WN = 1;                   // 32-row weight tiles a wave
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
      copy16(wp[i] + off, lds_address(S + (i * PASS + wid * 8) * MOE_BKB));
    else
      copy16(ap[i - 4] + off,
             lds_address(S + (TN + (i - 4) * PASS + wid * 8) * MOE_BKB));
  };
  auto offset = [&](int kt) {
    return min(kt * MOE_BKB + src * 16, p.kb - 16);
  };
  auto issue = [&](int kt, uint8_t* S) {
    const int off = offset(kt);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) copy(i, off, S);
  };

  const int wb = wid * 32;  // a wave takes 32 weight rows and all TM rows
  const int swz_l = (l31 >> 1) & 7;
  using frag_t = std::conditional_t<FP8, i32x8v, bf16x8v>;
  f32x16v acc[WN][WM] = {};

  // FULL: 128 bytes of the contraction; else what is left of it (32 k bytes).
  auto stage = [&](const uint8_t* S, int left, auto full, auto&& between) {
    constexpr bool FULL = decltype(full)::value;
    constexpr int KS = FP8 ? 2 : 4;
    const uint8_t* Wl = S + (wb + l31) * MOE_BKB;
    const uint8_t* Al = S + (TN + l31) * MOE_BKB;
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

  store_results<FP8, GATE>(p, acc, e, row0, rows_end, n0, wb);
}

// ---- many rows -----------------------------------------------------------------
// A workgroup takes up to 256 rows of one expert and 256 of its weight rows, 8 waves
// of 64 weight rows (4 across) and every other block of 32 rows (2 across): WM blocks
// of each, so that an expert's last tile costs what its rows do, in steps of 64.
// Operands lie in a ring of five units of 32 KB, a stage's W or A each: of turn t
// W is unit 2t, A unit 2t + 1, and W of turn t + 1 has had a turn longer to land.
// What bounds it: the card's power, and where operands come from behind the L2 the
// wait for them. 128 bf16 experts of 2048 x 768, 8192 tokens x 8: gate/up 443 us = 930
// TFLOP/s, down 2 x 159 us (tiles of 128 x 256, 48 KB a stage for half the products:
// 498 and 2 x 187), on other cards up to 498 and 2 x 168; with operands from the L2 alone 1.27 PFLOP/s, where the matrix
// cores work 88% of the cycles of a clock that sinks to 1.45 GHz: half the copies, or
// reads of LDS left out, raise the clock, not the products a cycle. Copies asked for in
// one burst hold their wave up, so they are spread over the products. Workgroups that
// go on to another block by a queue, so that the last ones end together, were no faster
// (of one run, a whole call: 870 us, 874 without), nor was a longer part of the chip busy.
// ---- its results: rows through LDS, so that a wave stores long runs of each --------
// Stored from the accumulators, 16 or 32 bytes of 32 rows an instruction: gate/up 351 /
// 325 us, down 143 / 122 (65,536 rows of one expert).

// Row block j of a wave: rows ab + 64 j + l31 of the tile. rowc, roww, rows_a: the
// choice, routing weight and activation scale of this thread's row (tid < 256).
template <bool FP8, bool GATE, int WM>
DEVINL void store_big(const MoeArgs& p, uint8_t* S, const f32x16v (&acc)[2][WM],
                      const int e, const int row0, const int rows, const int n0,
                      const int wb, const int ab, const int rowc,
                      const float roww, const float rows_a) {
  constexpr int PITCH = 272;  // bytes a row: 128 bf16 or 64 fp32, and 16
  const int tid = threadIdx.x;
  const int lane = tid & 63, l31 = lane & 31, half = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  int* choices = reinterpret_cast<int*>(S + 8 * 64 * PITCH);
  float* weights = reinterpret_cast<float*>(choices + 256);
  float* scales = weights + 256;
  __syncthreads();  // every wave is done with the ring
  if (tid < 256) {
    choices[tid] = rowc;
    weights[tid] = roww;
    if (FP8) scales[tid] = rows_a;
  }
  __syncthreads();
  if constexpr (GATE) {
#pragma unroll
    for (int j = 0; j < WM; ++j) {
      const int r = ab + j * 64 + l31;
      const float w = weights[r];
      const float sa = FP8 ? scales[r] : 1.f;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int f = (wb >> 1) + i * 16 + 8 * q + 4 * half;  // of the tile's 128
          const int fn = min(n0 + f, p.N - 4);  // not stored from N on
          f32x4v g, u;
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            g[s] = acc[i][j][4 * q + s];
            u[s] = acc[i][j][8 + 4 * q + s];
          }
          if (FP8) {
            const float* ws = p.w_scale + (size_t)e * 2 * p.N + fn;
            g *= sa * *reinterpret_cast<const f32x4v*>(ws);
            u *= sa * *reinterpret_cast<const f32x4v*>(ws + p.N);
          }
          if (p.in_w) {
            g *= w;
            u *= w;
          }
          if (p.bias != nullptr) {
            const uint16_t* b = p.bias + (size_t)e * 2 * p.N + fn;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
              g[s] += bf16_bits_to_f32(b[s]);
              u[s] += bf16_bits_to_f32(b[p.N + s]);
            }
          }
          float v[4];
          activate(p.limit, p.gelu, g, u, v);
          *reinterpret_cast<uint2*>(S + r * PITCH + f * 2) =
              make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
        }
    }
    __syncthreads();
    const int f = (tid & 15) * 8;
    uint16_t* h = (uint16_t*)p.out + (size_t)row0 * p.N + n0 + f;
    if (n0 + f < p.N)
#pragma unroll
      for (int k = 0; k < 2 * WM; ++k) {
        const int r = k * 32 + (tid >> 4);
        if (r < rows)
          *reinterpret_cast<int4*>(h + (size_t)r * p.N) =
              *reinterpret_cast<const int4*>(S + r * PITCH + f * 2);
      }
  } else {
    // a wave's own 64 rows of 64 features, twice
    uint8_t* T = S + wid * 64 * PITCH;
    float* y = (float*)p.out + n0 + wb - p.first;
    f32x4v ws[2][4];
    if (FP8)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          ws[i][q] = *reinterpret_cast<const f32x4v*>(
              p.w_scale + (size_t)e * p.N +
              min(n0 + wb + i * 32 + 8 * q + 4 * half, p.N - 4));
#pragma unroll
    for (int j0 = 0; j0 < WM; j0 += 2) {
#pragma unroll
      for (int j = j0; j < WM && j < j0 + 2; ++j) {
        const float w = weights[ab + j * 64 + l31];
        const float sa = FP8 ? scales[ab + j * 64 + l31] : 1.f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            f32x4v o;
#pragma unroll
            for (int s = 0; s < 4; ++s) o[s] = acc[i][j][4 * q + s];
            if (FP8) o *= w * (sa * ws[i][q]);
            else o *= w;
            *reinterpret_cast<f32x4v*>(T + ((j - j0) * 32 + l31) * PITCH +
                                       (i * 32 + 8 * q + 4 * half) * 4) = o;
          }
      }
      __builtin_amdgcn_wave_barrier();
      const int f = (lane & 15) * 4;
      if (n0 + wb + f < p.first + p.cols)
#pragma unroll
        for (int k = 0; k < (WM - j0 < 2 ? 8 : 16); ++k) {
          const int t = k * 4 + (lane >> 4);
          const int r = ab + (j0 + (t >> 5)) * 64 + (t & 31);
          if (r < rows)
            *reinterpret_cast<f32x4v*>(y + (size_t)choices[r] * p.cols + f) =
                *reinterpret_cast<const f32x4v*>(T + t * PITCH + f * 4);
        }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

template <bool FP8, bool GATE, int WM>
DEVINL void big_tile(const MoeArgs& p, uint8_t* S, const int e, const int row0,
                     const int rows_end, const int n0) {
  constexpr int WN = 2;
  constexpr int KS = FP8 ? 2 : 4;  // products along a stage
  constexpr int NB = FP8 ? 1 : 2;  // fp8: two sets of operands do not fit 256 registers
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  const int l31 = lane & 31;

  int rowc = 0;
  float roww = 1.f, rows_a = 1.f;
  if (tid < rows_end - row0 && tid < 256) {
    rowc = p.perm[row0 + tid];
    if (FP8) rows_a = p.a_scale[GATE ? rowc / p.topk : row0 + tid];
    if (GATE ? p.in_w : !p.in_w) roww = p.choice_w[rowc];
  }
  // ---- what a thread copies: one chunk of rows tid / 8 + 64 i, those of a wave from a
  // uniform row on (but the gathered rows of x)
  const int src = ((tid & 7) ^ ((tid >> 4) & 7)) * 16;
  const int r0 = wid * 8, lr = lane >> 3;
  const uint8_t* wp[4];
  uint32_t wo[4];
  const uint8_t* ap[WM];
  uint32_t ao[WM];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = i * 64 + r0;
    // rows past the last feature are read twice and never stored
    const int n = GATE ? n0 + (r >> 5) * 16 + (r & 15) : n0 + r;
    const int n1 = min(n, p.N - 1);
    const int row = n1 + (GATE ? ((r >> 4) & 1) * p.N : 0);
    wp[i] = p.w + ((size_t)e * (GATE ? 2 * p.N : p.N) + row) * p.kb;
    wo[i] = (uint32_t)min(lr, p.N - 1 - n1) * (uint32_t)p.kb + src;
  }
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int r = min(row0 + i * 64 + r0, rows_end - 1);
    const int l = min(lr, rows_end - 1 - r);
    ap[i] = p.a + (GATE ? (size_t)(p.perm[r + l] / p.topk) * p.kb + src
                        : (size_t)r * p.kb);
    ao[i] = (uint32_t)l * (uint32_t)p.kb + src;
  }
  const uint32_t s0 = lds_address(S) + r0 * MOE_BKB;
  auto copy_w = [&](int i, int off, int u) {
    copy16(wp[i] + off, wo[i], s0 + u * MOE_UNIT + i * 64 * MOE_BKB);
  };
  auto copy_a = [&](int i, int off, int u) {
    const uint32_t at = s0 + u * MOE_UNIT + i * 64 * MOE_BKB;
    if (GATE) copy16(ap[i] + off, at);
    else copy16(ap[i] + off, ao[i], at);
  };
  auto issue_w = [&](int off, int u) {
#pragma unroll
    for (int i = 0; i < 4; ++i) copy_w(i, off, u);
  };
  auto issue_a = [&](int off, int u) {
#pragma unroll
    for (int i = 0; i < WM; ++i) copy_a(i, off, u);
  };
  const int nk = p.kb / MOE_BKB;  // full stages
  // Past the last full stage the copies go on, of that stage again, so that their
  // number in flight is the same for every turn and the wait a constant.
  auto offset = [&](int kt) { return min(kt, nk - 1) * MOE_BKB; };

  const int wb = (wid & 3) * 64, ab = (wid >> 2) * 32;
  const int swz_l = (l31 >> 1) & 7;
  using frag_t = std::conditional_t<FP8, i32x8v, bf16x8v>;
  f32x16v acc[WN][WM] = {};
  frag_t a[NB][WN], b[NB][WM];
  // of units u (W) and v (A); left: bytes of the contraction in the stage
  auto fetch = [&](int u, int v, int ks, int left, auto full) {
    constexpr bool FULL = decltype(full)::value;
    const uint8_t* W = S + u * MOE_UNIT;
    const uint8_t* A = S + v * MOE_UNIT;
#pragma unroll
    for (int i = 0; i < WN + WM; ++i) {
      const uint8_t* r = i < WN ? W + (wb + i * 32 + l31) * MOE_BKB
                                : A + (ab + (i - WN) * 64 + l31) * MOE_BKB;
      frag_t& f = i < WN ? a[ks % NB][i] : b[ks % NB][i - WN];
      if constexpr (FP8) {
        const int c0 = ((4 * ks + 2 * half) ^ swz_l) * 16;
        const int c1 = ((4 * ks + 2 * half + 1) ^ swz_l) * 16;
        f = __builtin_shufflevector(*(const i32x4v*)(r + c0),
                                    *(const i32x4v*)(r + c1), 0, 1, 2, 3, 4, 5,
                                    6, 7);
        // of a last step of 32 the upper half of the lanes has nothing, and of
        // a step behind the end no lane has
        if (!FULL && left - ks * 64 < (half ? 64 : 1)) f = 0;
      } else {
        f = *(const bf16x8v*)(r + ((2 * ks + half) ^ swz_l) * 16);
        if (!FULL && ks * 32 >= left) f = 0;
      }
    }
  };
  auto products = [&](int ks, auto&& between) {
#pragma unroll
    for (int i = 0; i < WN; ++i)
#pragma unroll
      for (int j = 0; j < WM; ++j) {
        if constexpr (FP8)
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
              a[ks % NB][i], b[ks % NB][j], acc[i][j], 0, 0, 0, 0x7f7f7f7f, 0,
              0x7f7f7f7f);
        else
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              a[ks % NB][i], b[ks % NB][j], acc[i][j], 0, 0, 0);
        between(i * WM + j);
      }
  };
  // lgkmcnt(0) before the next step's operands are asked for: this step's products
  // need no further wait and run while those are under way
  auto landed = [] {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_sched_barrier(0);
  };
  // a fence would wait for every copy: vmcnt(V) and lgkmcnt(0) by hand, and no LDS
  // access moves over the barrier
  auto meet = [](auto v) {
    constexpr int V = decltype(v)::value;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070 | (V & 15) | ((V >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // A copy between products: a wave that asks for several at once waits for the
  // address unit, which takes 64 bytes a cycle.
  auto spread = [](int m, int first, int step, int n, auto&& copy) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < n && m == first + i * step) {
        __builtin_amdgcn_sched_barrier(0);
        copy(i);
        __builtin_amdgcn_sched_barrier(0);
      }
  };

  // Turn kt: products of units u (W) and u + 1 (A); the copies of W two turns on go
  // to u + 4. Before the last products every wave has its operands in registers:
  // behind that barrier the next turn's units are there, and A two turns on goes to
  // W's own place.
  auto turn = [&](int kt, auto unit) {
    constexpr int u = decltype(unit)::value;
    const int off = offset(kt + 2);
    constexpr int PRODUCTS = WN * WM;
    constexpr int STEP = (KS - 1) * PRODUCTS / 4;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      auto next = [&] {
        if (ks + 1 < KS) fetch(u, (u + 1) % 5, ks + 1, MOE_BKB, std::true_type{});
        else fetch((u + 2) % 5, (u + 3) % 5, 0, MOE_BKB, std::true_type{});
        __builtin_amdgcn_sched_barrier(0);
      };
      landed();
      if (ks + 1 == KS) meet(std::integral_constant<int, 4>{});
      if (NB == 2) next();
      products(ks, [&](int m) {
        if (ks + 1 < KS)
          spread(ks * PRODUCTS + m, 0, STEP, 4,
                 [&](int i) { copy_w(i, off, (u + 4) % 5); });
        else
          spread(m, 0, PRODUCTS / WM, WM, [&](int i) { copy_a(i, off, u); });
      });
      if (NB == 1) next();
    }
  };
  if (nk > 0) {
    issue_w(0, 0);
    issue_a(0, 1);
    issue_w(offset(1), 2);
    issue_a(offset(1), 3);
    meet(std::integral_constant<int, 4 + WM>{});
    fetch(0, 1, 0, MOE_BKB, std::true_type{});
    for (int kt = 0; kt < nk;) {
      turn(kt, std::integral_constant<int, 0>{});
      if (++kt >= nk) break;
      turn(kt, std::integral_constant<int, 2>{});
      if (++kt >= nk) break;
      turn(kt, std::integral_constant<int, 4>{});
      if (++kt >= nk) break;
      turn(kt, std::integral_constant<int, 1>{});
      if (++kt >= nk) break;
      turn(kt, std::integral_constant<int, 3>{});
      ++kt;
    }
    // the last copies: no more may land in LDS once the workgroup has ended
    __builtin_amdgcn_s_waitcnt(0x0070);
  }
  const int left = p.kb % MOE_BKB;
  if (left) {
    __syncthreads();
    const int back = max(src - (left - 16), 0);  // within the row
    const int at = nk * MOE_BKB;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      copy16(wp[i] + at, wo[i] - back, s0 + i * 64 * MOE_BKB);
#pragma unroll
    for (int i = 0; i < WM; ++i)
      copy16(ap[i] + at + (GATE ? 0 : ao[i]) - back,
             s0 + MOE_UNIT + i * 64 * MOE_BKB);
    meet(std::integral_constant<int, 0>{});
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      fetch(0, 1, ks, left, std::false_type{});
      products(ks, [](int) {});
    }
  }
  store_big<FP8, GATE, WM>(p, S, acc, e, row0, rows_end - row0, n0, wb, ab, rowc,
                           roww, rows_a);
}

template <bool FP8, bool GATE>
__global__ __launch_bounds__(512, 2) void moe_big_kernel(const MoeArgs p) {
  __shared__ __attribute__((aligned(128))) uint8_t S[5 * MOE_UNIT];
  // an eighth of the list an XCD, see moe_gemm_kernel
  const int total = *p.n_tiles * p.nb;
  const int chunk = (total + 7) >> 3;
  const int slot = blockIdx.x >> 3;
  const int idx = (blockIdx.x & 7) * chunk + slot;
  if (slot >= chunk || idx >= total) return;
  const int4 tile = p.tiles[idx / p.nb];
  const int e = __builtin_amdgcn_readfirstlane(tile.x);
  const int row0 = __builtin_amdgcn_readfirstlane(tile.y);
  const int rows_end = __builtin_amdgcn_readfirstlane(tile.z);
  const int n0 = p.first + (idx % p.nb) * (GATE ? 128 : 256);
  const int rows = rows_end - row0;
  if (rows > 192)
    big_tile<FP8, GATE, 4>(p, S, e, row0, rows_end, n0);
  else if (rows > 128)
    big_tile<FP8, GATE, 3>(p, S, e, row0, rows_end, n0);
  else if (rows > 64)
    big_tile<FP8, GATE, 2>(p, S, e, row0, rows_end, n0);
  else
    big_tile<FP8, GATE, 1>(p, S, e, row0, rows_end, n0);
}
// ---- combine --------------------------------------------------------------------
// out[t] = sum over its choices, of the features from first on; four a thread. Memory
// bounds it (5.2 TB/s of y), a round trip or two with few tokens: a ballot tells which
// choices have rows, those of experts of other ranks have none, and up to eight rows are
// loaded at once, with fewer left four or two. us of the kernel, a load and an addition
// in turn / all choices loaded, those without rows too / so: 8,192 tokens of 8 choices,
// 2048 features, all experts here 106.8 / 102.4 / 103.2, one in eight 23.3 / 87.5 / 22.3;
// 24 tokens 4.8 / 4.2 / 4.2; 8,192 of 2 choices, 1024 features, 15.6 / 15.0 / 15.9 and 8.0
// / 10.3 / 8.7. The mask from scalar loads of the ids: one in eight 26.7, two choices
// 15.6 and 8.4.

// adds the rows of the first C choices of the mask and takes them off it
template <int C>
DEVINL void add_choices(f32x4v& s, const float* y, int cols, u64& mask) {
  const int n = __popcll(mask);
  uint32_t row = 0;
  f32x4v v[C];
  asm volatile("; up to %0" ::"n"(C) : "memory");  // no loads shared between the sizes
#pragma unroll
  for (int i = 0; i < C; ++i) {  // past the last one that one again
    row = mask ? __ffsll(mask) - 1 : row;
    mask &= mask - 1;
    v[i] = *reinterpret_cast<const f32x4v*>(y + row * (uint32_t)cols);
  }
#pragma unroll
  for (int i = 0; i < C; ++i)
    if (i < n) s += v[i];
}

__global__ __launch_bounds__(256) void moe_combine_kernel(
    float* __restrict__ out, const float* __restrict__ y,
    const int64_t* __restrict__ ids, const int T, const int k, const int E,
    const int H, const int first, const int cols) {
  const int t = blockIdx.x, lane = threadIdx.x & 63;
  auto local = [&](int j0) {  // of choices j0 .. j0 + 63, those of experts that are here
    const int64_t e = j0 + lane < k ? ids[(size_t)t * k + j0 + lane] : -1;
    return (u64)__ballot(e >= 0 && e < E);
  };
  const u64 all = local(0);
  for (int c0 = blockIdx.y * 1024; c0 < cols; c0 += gridDim.y * 1024) {
    const int c = c0 + threadIdx.x * 4;
    const float* row = y + (size_t)t * k * cols + min(c, cols - 4);
    f32x4v s = {0.f, 0.f, 0.f, 0.f};
    for (int j0 = 0; j0 < k; j0 += 64, row += (size_t)64 * cols)
      for (u64 mask = j0 ? local(j0) : all; mask;) {
        const int n = __popcll(mask);
        if (n > 4) add_choices<8>(s, row, cols, mask);
        else if (n > 2) add_choices<4>(s, row, cols, mask);
        else add_choices<2>(s, row, cols, mask);
      }
    if (c < cols) *reinterpret_cast<f32x4v*>(out + (size_t)t * H + first + c) = s;
  }
}

extern "C" void launch_quantize_fp8_rows(
    void* out, float* scales, const void* x, int R, int C,
    hipStream_t stream) {
  quantize_fp8_rows_kernel<<<R, 256, 0, stream>>>(
      (uint8_t*)out, scales, (const uint16_t*)x, C);
}

// ---- the two products of a layer -----------------------------------------------

template <bool FP8, int TM, int STAGES>
static void launch_gemm(bool gate, MoeArgs& p, int max_tiles,
                        hipStream_t stream) {
  p.nb = ceil_div(p.cols, gate ? 64 : 128);
  const int blocks = (max_tiles * p.nb + 7) / 8 * 8;
  if (gate)
    moe_gemm_kernel<FP8, TM, true, STAGES><<<blocks, 256, 0, stream>>>(p);
  else
    moe_gemm_kernel<FP8, TM, false, STAGES><<<blocks, 256, 0, stream>>>(p);
}

template <bool FP8>
static void launch_gemm_tm(int tm, bool gate, MoeArgs& p, int max_tiles,
                           hipStream_t stream) {
  if (tm == 32) {
    launch_gemm<FP8, 32, 4>(gate, p, max_tiles, stream);
  } else if (tm == 64) {
    launch_gemm<FP8, 64, 3>(gate, p, max_tiles, stream);
  } else {
    p.nb = ceil_div(p.cols, gate ? 128 : 256);
    const int blocks = (max_tiles * p.nb + 7) / 8 * 8;
    if (gate) {
      moe_big_kernel<FP8, true><<<blocks, 512, 0, stream>>>(p);
    } else {
      moe_big_kernel<FP8, false><<<blocks, 512, 0, stream>>>(p);
    }
  }
}

// Rows a tile, by the mean number of choices an expert and by how many blocks of 256
// rows x 256 weight rows there are: fewer than CUs leave some of them idle, unless the
// experts' last tiles are few beside the full ones. Measured (us, tiles of 32 / 64 /
// 256 rows): bf16 128 experts of 2048 x 768, mean 6: 180 / 181 / 201, 25: 247 / 241 /
// 241, 50: 319 / 289 / 284, 100: 456 / 379 / 340, 300: 1091 / 815 / 608; 32 experts of
// 2048 x 1024, mean 50: 124 / 115 / 128, 125: 191 / 157 / 168 (240 blocks), 150: 231 /
// 169 / 164 (280), 400: 504 / 360 / 280; 16 experts of 1024 x 512, mean 300: 58 / 57 /
// 67 (104), 625: 104 / 87 / 78 (188); fp8 256 experts of 7168 x 2048, mean 2: 961 / 961
// / 984, 6: 1432 / 1415 / 1389, 25: 2177 / 1881 / 1739, 47: 3228 / 2409 / 2028; 128 of
// 2048 x 768, mean 12: 131 / 131 / 135, 25: 155 / 156 / 151, 200: 492 / 424 / 346.
extern "C" int moe_tile_rows(int n, int E, int I, bool fp8) {
  const int mean = n / (E > 0 ? E : 1);
  const int64_t blocks = ((int64_t)n / 256 + E / 2) * ceil_div(I, 128);
  if (mean > 450 || (blocks >= 256 && mean > (fp8 ? 16 : 40)) ||
      (fp8 && blocks >= 2048 && mean > 4))
    return 256;
  return mean <= (fp8 ? 12 : 24) ? 32 : 64;
}

extern "C" int moe_max_tiles(int n, int E, int tm) {
  return n / tm + (n < E ? n : E);
}

// Output features of a down product and combine: y takes at most MOE_Y_BYTES (of
// 256 features, a tile's width, at least), however many tokens a step brings. 65,536
// choices of 2048 features, a whole call with the tiles of 128 rows that there were:
// one slab of 537 MB 1.033 ms, two of 256 MB at most 1.030; now with 512 / 256 / 128 MB
// 900 / 892 / 905 us, 40,000 choices 603 / 609 / 618, 16,000 366 / 361 / 361.
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

// xq not null: x's rows are quantised too
extern "C" void launch_moe_route(int* perm, void* tiles, int* n_tiles,
                                 int* counts, const int64_t* ids, int n, int E,
                                 int tm, void* xq, float* xs, const void* x, int T,
                                 int H, hipStream_t stream) {
  const int parts = route_parts(n, E);
  const QuantizeRows rows{(uint8_t*)xq, xs, (const uint16_t*)x, T, H};
  const int more = xq != nullptr ? ceil_div(T, ROUTE_THREADS / 256) : 0;
  if (E > ROUTE_LDS) {
    moe_route_kernel<false><<<1 + more, ROUTE_THREADS, 0, stream>>>(
        perm, (int4*)tiles, n_tiles, counts, ids, n, E, tm, 1, rows);
    return;
  }
  if (parts > 1)
    moe_count_kernel<<<parts, ROUTE_THREADS, E * sizeof(int), stream>>>(
        counts, ids, n, E);
  moe_route_kernel<true><<<parts + more, ROUTE_THREADS, E * sizeof(int), stream>>>(
      perm, (int4*)tiles, n_tiles, counts, ids, n, E, tm, parts, rows);
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
  moe_combine_kernel<<<grid, 256, 0, stream>>>(out, y, ids, T, k, E, H, first, cols);
}
