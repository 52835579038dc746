// Routed experts of at most 32 choices, in two launches: the decode step of one or a few
// requests (moe_few_takes has the sizes).
//
//   moe_few_gate   h[choice] = act(x[token] . W_gu[e]^T), 16 features of one expert a
//                  workgroup, whose waves share K
//   moe_few_down   out[token] = sum over its choices of w (h[choice] . W_down[e]^T),
//                  fp32, eight or 16 features of every expert a workgroup, whose waves
//                  share the list of the experts' steps along K
//
// What bounds it: the launches and two memory round trips each, and from a dozen experts
// on their weights' stream. Every choice is a lane's, so that each wave finds its expert
// and that one's rows by ballots: no launch sorts them, and as a token's choices meet in
// one workgroup none adds them up. Rows go eight at a time; an expert of more is read
// again for the next eight.
//
// A call, us, the kernels for more choices (moe.hip) / these, of 1, 2, 4 and 8 tokens: 32
// experts of 2048 x 1024, 4 a token, 24.6 / 16.3, 25.9 / 21.1, 31.7 / 29.1, 58.3 / 48.6, in
// fp8 30.3 / 21.8, 30.1 / 22.6, 30.4 / 27.5, 35.1 / 35.4; 128 of 2048 x 768, 8 a token, 26.7
// / 22.5, 36.4 / 36.7, 65.4 / 60.9, in fp8 29.7 / 22.8, 32.1 / 30.8, 43.3 / 44.1; 16 of
// 1024 x 512, 2 a token, 20.5 / 12.7 of 1 token, 20.2 / 14.5 of 8, 20.3 / 17.6 of 16; fp8,
// 256 of 7168 x 2048, 8 a token, 82 / 81, of 2 tokens 140 / 143.
#include <cmath>
#include <type_traits>

#include "moe_common.h"

#define FEW_N 32         // choices
#define FEW_ROWS 8       // of an expert at a time
#define FEW_SPAN 128     // bytes along K of a stage
#define FEW_GATE_WAVES 4

struct FewArgs {
  const uint8_t* w;        // gate: [E, 2 N, kb] bytes, down: [E, N, kb]
  const float* w_scale;    // of its rows (fp8)
  const uint8_t* a;        // gate: x [T, kb], down: h [n, kb]
  const float* a_scale;    // of its rows (fp8)
  const int64_t* ids;      // [n]
  const float* choice_w;   // [n]
  const uint16_t* bias;    // [E, 2 N] or null (gate)
  void* out;               // gate: h [n, N] bf16, down: [T, N] fp32
  int n, topk, E, N, kb;
  int in_w, gelu;
  float limit;
};

namespace {

typedef unsigned long long u64;

template <int N>
DEVINL void wait_copies() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N & 48) << 10));
  asm volatile("" ::: "memory");
}

// this wave's operands are in registers, and what follows stays behind
DEVINL void landed() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_sched_barrier(0);
}

// a lane's expert, -1 for those of other ranks
DEVINL int expert_of(const FewArgs& p) {
  const int lane = threadIdx.x & 63;
  const int64_t id = lane < p.n ? p.ids[lane] : -1;
  return id >= 0 && id < p.E ? (int)id : -1;
}

// The j-th of the choices in `mask`, the last one where there are fewer; j < 8.
DEVINL int nth(u64 mask, int j) {
#pragma unroll
  for (int i = 0; i < FEW_ROWS - 1; ++i) {
    const u64 rest = mask & (mask - 1);
    mask = i < j && rest ? rest : mask;
  }
  return __ffsll(mask) - 1;
}

// the choices behind the first eight
DEVINL u64 behind(u64 mask) {
#pragma unroll
  for (int i = 0; i < FEW_ROWS; ++i) mask &= mask - 1;
  return mask;
}

// 16 x 16 products of one stage: rows `a` of LDS (of W) and `b` (activations), whose
// 16-byte chunk j lies at j ^ (row / 2 & 7)
template <bool FP8, int AT>
struct Operands {
  bf16x8v a[2][AT], b[2];
  DEVINL void fetch(const uint8_t* S, const int (&ra)[AT], int rb) {
    const int l4 = (threadIdx.x >> 4) & 3;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int c = l4 + 4 * k;
#pragma unroll
      for (int t = 0; t < AT; ++t)
        a[k][t] = *reinterpret_cast<const bf16x8v*>(
            S + ra[t] * FEW_SPAN + (c ^ ((ra[t] >> 1) & 7)) * 16);
      b[k] = *reinterpret_cast<const bf16x8v*>(S + rb * FEW_SPAN +
                                               (c ^ ((rb >> 1) & 7)) * 16);
    }
  }
  static DEVINL i32x8v join(bf16x8v lo, bf16x8v hi) {
    return __builtin_shufflevector(__builtin_bit_cast(i32x4v, lo),
                                   __builtin_bit_cast(i32x4v, hi), 0, 1, 2, 3, 4, 5, 6, 7);
  }
  DEVINL void multiply(f32x4v (&acc)[AT]) const {
#pragma unroll
    for (int t = 0; t < AT; ++t) {
      if constexpr (FP8) {
        acc[t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
            join(a[0][t], a[1][t]), join(b[0], b[1]), acc[t], 0, 0, 0, 0x7f7f7f7f, 0,
            0x7f7f7f7f);
      } else {
#pragma unroll
        for (int k = 0; k < 2; ++k)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[k][t], b[k], acc[t], 0, 0, 0);
      }
    }
  }
};

}  // namespace

// Workgroup (16 features, the d-th expert in the order of the choices). A wave has its
// own ring of stages, of 16 gate rows, 16 up rows and 8 rows of x.
template <bool FP8>
__global__ __launch_bounds__(FEW_GATE_WAVES * 64, 2) void moe_few_gate_kernel(
    const FewArgs p) {
  constexpr int WAVES = FEW_GATE_WAVES, STAGES = 4, NI = 5;
  constexpr int RING = (32 + FEW_ROWS) * FEW_SPAN;
  __shared__ __attribute__((aligned(128))) uint8_t S[WAVES * STAGES * RING];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l4 = lane >> 4;
  const int id = expert_of(p);
  u64 left = __ballot(id >= 0), mask;
  int e;
  for (int d = blockIdx.y;; --d) {
    if (left == 0) return;
    e = __builtin_amdgcn_readlane(id, __ffsll(left) - 1);
    mask = __ballot(id == e);
    if (d == 0) break;
    left &= ~mask;
  }
  const int n0 = blockIdx.x * 16;
  const uint8_t* wb = p.w + (size_t)e * 2 * p.N * p.kb;
  uint32_t at[NI];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = q * 8 + (lane >> 3);
    // rows past the last feature are read twice and never stored
    at[q] = (uint32_t)(min(n0 + (r & 15), p.N - 1) + (r >> 4) * p.N) * p.kb +
            ((lane & 7) ^ ((r >> 1) & 7)) * 16;
  }
  const int cols = p.kb / FEW_SPAN;
  const int mine = (cols - wid + WAVES - 1) / WAVES;
  uint8_t* ring = S + wid * (STAGES * RING);
  const uint32_t ring_at = lds_address(ring);
  const int ra[2] = {l15, 16 + l15}, rb = 32 + (l15 & 7);
  float* part = reinterpret_cast<float*>(S);  // [wave][row][32]

  for (; mask; mask = behind(mask)) {
    const int rows = min(__popcll(mask), FEW_ROWS);
    at[4] = (uint32_t)(nth(mask, lane >> 3) / p.topk) * (uint32_t)p.kb +
            ((lane & 7) ^ (((32 + (lane >> 3)) >> 1) & 7)) * 16;
    auto issue = [&](int i, int place) __attribute__((always_inline)) {
      const int k = (min(i, mine - 1) * WAVES + wid) * FEW_SPAN;
#pragma unroll
      for (int q = 0; q < NI; ++q)
        copy16((q < 4 ? wb : p.a) + k, at[q], ring_at + place * RING + q * 1024);
    };
    f32x4v acc[2] = {};
    if (mine > 0) {
#pragma unroll
      for (int i = 0; i < STAGES - 1; ++i) issue(i, i);
      int place = 0, next = STAGES - 1;
      for (int i = 0; i < mine; ++i) {
        wait_copies<(STAGES - 2) * NI>();
        Operands<FP8, 2> o;
        o.fetch(ring + place * RING, ra, rb);
        landed();
        issue(i + STAGES - 1, next);  // the place of the turn before
        o.multiply(acc);
        place = place + 1 == STAGES ? 0 : place + 1;
        next = next + 1 == STAGES ? 0 : next + 1;
      }
      wait_copies<0>();
    }
    __syncthreads();
    if (l15 < FEW_ROWS)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        *reinterpret_cast<f32x4v*>(part + (wid * FEW_ROWS + l15) * 32 + t * 16 + l4 * 4) =
            acc[t];
    __syncthreads();
    const int row = tid >> 2, f = (tid & 3) * 4, fn = min(n0 + f, p.N - 4);
    if (row < rows && n0 + f < p.N) {
      f32x4v g = {}, u = {};
#pragma unroll
      for (int v = 0; v < WAVES; ++v) {
        g += *reinterpret_cast<const f32x4v*>(part + (v * FEW_ROWS + row) * 32 + f);
        u += *reinterpret_cast<const f32x4v*>(part + (v * FEW_ROWS + row) * 32 + 16 + f);
      }
      const int choice = nth(mask, row);
      if (FP8) {
        const float sa = p.a_scale[choice / p.topk];
        const float* ws = p.w_scale + (size_t)e * 2 * p.N + fn;
        g *= sa * *reinterpret_cast<const f32x4v*>(ws);
        u *= sa * *reinterpret_cast<const f32x4v*>(ws + p.N);
      }
      if (p.in_w) {
        const float w = p.choice_w[choice];
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
      *reinterpret_cast<uint2*>((uint16_t*)p.out + (size_t)choice * p.N + n0 + f) =
          make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
    }
    __syncthreads();  // the ring is filled again
  }
}

// Workgroup: NT features, all experts. A unit is up to eight choices of one expert;
// the stages of all units form one list, of which every wave takes an equal run. A
// wave's sums go to its own table of tokens where a unit ends.
template <bool FP8, int NT, int STAGES>
__global__ __launch_bounds__(512, 2) void moe_few_down_kernel(const FewArgs p) {
  constexpr int WAVES = 8, NI = NT / 8 + 1;
  constexpr int RING = (NT + FEW_ROWS) * FEW_SPAN;
  __shared__ __attribute__((aligned(128))) uint8_t S[WAVES * STAGES * RING];
  __shared__ float table[WAVES][FEW_N][NT];  // [wave][token][feature]
  __shared__ int unit_e[FEW_N], unit_rows[FEW_N], units;
  __shared__ int unit_c[FEW_N][FEW_ROWS], unit_t[FEW_N][FEW_ROWS];  // choices, tokens
  __shared__ float unit_w[FEW_N][FEW_ROWS], unit_s[FEW_N][NT];  // factors of both
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l4 = lane >> 4;
  const int n0 = blockIdx.x * NT;
  const int tokens = p.n / p.topk;
  if (wid == 0) {
    const int id = expert_of(p);
    const int own = min(lane, p.n - 1);
    const float w = (p.in_w ? 1.f : p.choice_w[own]) * (FP8 ? p.a_scale[own] : 1.f);
    const int token = own / p.topk;
    u64 left = __ballot(id >= 0);
    int u = 0;
    while (left) {
      const int e = __builtin_amdgcn_readlane(id, __ffsll(left) - 1);
      u64 mask = __ballot(id == e);
      left &= ~mask;
      for (; mask; mask = behind(mask)) {
        const int mine = nth(mask, lane & 7);
        const float f = __shfl(w, mine, WAVE_SIZE);
        const int t = __shfl(token, mine, WAVE_SIZE);
        if (lane < FEW_ROWS) {
          unit_c[u][lane] = mine;
          unit_t[u][lane] = t;
          unit_w[u][lane] = f;
        }
        if (lane == 0) {
          unit_e[u] = e;
          unit_rows[u] = min(__popcll(mask), FEW_ROWS);
        }
        ++u;
      }
    }
    if (lane == 0) units = u;
  }
  for (int i = tid; i < WAVES * FEW_N * NT; i += WAVES * 64) (&table[0][0][0])[i] = 0.f;
  __syncthreads();
  const int nu = __builtin_amdgcn_readfirstlane(units);
  if constexpr (FP8) {
    for (int i = tid; i < nu * NT; i += WAVES * 64)
      unit_s[i / NT][i % NT] =
          p.w_scale[(size_t)unit_e[i / NT] * p.N + min(n0 + i % NT, p.N - 1)];
    __syncthreads();
  }

  const int cols = p.kb / FEW_SPAN;
  const int total = nu * cols, per = (total + WAVES - 1) / WAVES;
  const int begin = wid * per, end = min(total, begin + per);
  uint8_t* ring = S + wid * (STAGES * RING);
  const uint32_t ring_at = lds_address(ring);
  const int r = lane >> 3;
  const uint32_t a_in = ((lane & 7) ^ (((NT + r) >> 1) & 7)) * 16;
  if (begin < end) {
    // the stage that is asked for next; at the run's end the last one again
    int s = begin, su = begin / cols, sc = begin % cols;
    const uint8_t *wp[NT / 8], *ap;
    auto enter = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < NT / 8; ++q)
        wp[q] = p.w + ((size_t)unit_e[su] * p.N + min(n0 + q * 8 + r, p.N - 1)) * p.kb +
                ((lane & 7) ^ (((q * 8 + r) >> 1) & 7)) * 16;
      ap = p.a + (size_t)unit_c[su][r] * p.kb + a_in;
    };
    enter();
    auto issue = [&](int place) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < NT / 8; ++q)
        copy16(wp[q] + sc * FEW_SPAN, ring_at + place * RING + q * 1024);
      copy16(ap + sc * FEW_SPAN, ring_at + place * RING + NT * FEW_SPAN);
      if (s + 1 < end) {
        ++s;
        if (++sc == cols) {
          sc = 0;
          ++su;
          enter();
        }
      }
    };
#pragma unroll
    for (int i = 0; i < STAGES - 1; ++i) issue(i);
    const int ra[1] = {l15 & (NT - 1)}, rb = NT + (l15 & 7);
    f32x4v acc[1] = {};
    int place = 0, next = STAGES - 1, u = begin / cols, col = begin % cols;
    for (int i = begin; i < end; ++i) {
      wait_copies<(STAGES - 2) * NI>();
      Operands<FP8, 1> o;
      o.fetch(ring + place * RING, ra, rb);
      landed();
      issue(next);  // the place of the turn before
      o.multiply(acc);
      place = place + 1 == STAGES ? 0 : place + 1;
      next = next + 1 == STAGES ? 0 : next + 1;
      if (++col == cols || i + 1 == end) {
        if (l15 < unit_rows[u] && l4 < NT / 4) {
          const float w = unit_w[u][l15];
          float* t = table[wid][unit_t[u][l15]] + l4 * 4;
#pragma unroll
          for (int f = 0; f < 4; ++f)  // a token may have chosen an expert twice
            atomicAdd(t + f, acc[0][f] * (FP8 ? w * unit_s[u][l4 * 4 + f] : w));
        }
        acc[0] = 0.f;
        col = 0;
        ++u;
      }
    }
    wait_copies<0>();
  }
  __syncthreads();
  for (int i = tid; i < tokens * NT; i += WAVES * 64) {
    const int t = i / NT, f = i % NT;
    if (n0 + f >= p.N) continue;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v += table[w][t][f];
    ((float*)p.out)[(size_t)t * p.N + n0 + f] = v;
  }
}

// Features of a workgroup of the second launch. Eight give the chip's 256 workgroups where
// H is 2048, and a workgroup's start is not paid twice: 7168 with 8 / 16 features 91 / 79 us,
// 2048 (32 choices) 48.6 / 52.1.
static int few_features(int H) { return H <= 2048 ? 8 : 16; }

// Up to 32 choices, in fp8, whose weights are half as much, 16 (see above; with room for
// 64, 40 / 48 / 64 choices took, general / these: 128 experts of 2048 x 768 76.1 / 77.2,
// 95.3 / 93.6, 107.8 / 111.5; fp8 24 / 32: 43.6 / 43.2, 45.0 / 50.1).
//
// Of these up to eight, and beyond the ones where two launches less, some 9 us, are worth
// more than what the small tiles cost: 0.3 to 0.4 us for each expert that is met, the
// choices being alike, and the time in which only a part of the chip reads the second
// launch's weights: where H gives few workgroups, or a few beyond a round. General / these:
// 32 of 128 experts of 256 x 768 23.2 / 37.6 (32 workgroups), of 512 x 128 16.6 / 21.8; 24
// of 64 of 4480 x 1280 147 / 160 (280 workgroups); 30 of 64 of 768 x 1024 32.4 / 44.4. Of
// 810 drawn sizes 130 were slower here, by up to 48%; of the 550 on this side of the line
// 14 are, by 3 to 12%, and they are 1.34 times as fast in the mean.
extern "C" bool moe_few_takes(int n, int E, int H, int I, bool fp8) {
  const int size = fp8 ? 1 : 2;
  if (n < 1 || n > (fp8 ? FEW_N / 2 : FEW_N) || E < 1 || H * size % FEW_SPAN ||
      I * size % FEW_SPAN || 2ll * I * H * size >= 1ll << 32)
    return false;
  const double met = E * (1. - std::pow(1. - 1. / E, n));
  const int nt = few_features(H), rounds = ceil_div(ceil_div(H, nt), 256);
  const double idle = (rounds * nt - H / 256.) * I * size * met;  // bytes a CU
  return n <= 8 || met + idle / 5000. <= 28.5;
}

extern "C" void launch_moe_few_gate(void* h, const void* x, const float* x_scale,
                                    const void* w, const float* w_scale,
                                    const int64_t* ids, const float* choice_w,
                                    const void* bias, int n, int topk, int E, int H, int I,
                                    bool fp8, bool in_w, bool gelu, float limit,
                                    hipStream_t stream) {
  const FewArgs p{(const uint8_t*)w, w_scale, (const uint8_t*)x, x_scale, ids, choice_w,
                  (const uint16_t*)bias, h, n, topk, E, I, fp8 ? H : 2 * H, in_w, gelu,
                  limit};
  const dim3 grid(ceil_div(I, 16), n < E ? n : E);
  auto run = [&](auto kernel) { kernel<<<grid, FEW_GATE_WAVES * 64, 0, stream>>>(p); };
  if (fp8) run(moe_few_gate_kernel<true>);
  else run(moe_few_gate_kernel<false>);
}

extern "C" void launch_moe_few_down(float* out, const void* h, const float* h_scale,
                                    const void* w, const float* w_scale,
                                    const int64_t* ids, const float* choice_w, int n,
                                    int topk, int E, int H, int I, bool fp8, bool in_w,
                                    hipStream_t stream) {
  const FewArgs p{(const uint8_t*)w, w_scale, (const uint8_t*)h, h_scale, ids, choice_w,
                  nullptr, out, n, topk, E, H, fp8 ? I : 2 * I, in_w, 0, 0.f};
  auto run = [&](auto kernel, int nt) { kernel<<<ceil_div(H, nt), 512, 0, stream>>>(p); };
  if (few_features(H) == 8) {
    if (fp8) run(moe_few_down_kernel<true, 8, 6>, 8);
    else run(moe_few_down_kernel<false, 8, 6>, 8);
  } else {
    if (fp8) run(moe_few_down_kernel<true, 16, 4>, 16);
    else run(moe_few_down_kernel<false, 16, 4>, 16);
  }
}
