// The layers of a Llama-type stack on a decode step of one to four requests, all in one
// launch: norm and q/k/v product, rope, cache and attention, output product, norm and
// gated product, down product, and so on through the layers.
//
// What bounds it: such a step is a chain of short products, each of which needs all of
// the one before. As launches of their own they take a memory round trip or two and the
// launch's ends each, far more than the weights' stream. Here a workgroup does a tile of
// one phase of one layer. It asks for its weights (or its part of the cache) first, when
// the phases before are still on their way, and then waits for its input; thus the
// weights of one to two layers are always underway, and a phase costs the way of its
// results to the next one's workgroups: about 3 us, half of it until they see them.
//
// That way is made of 64-bit words, 32 bits of value and 32 of a tag, the layer's number:
// one relaxed atomic store at device scope each, looked at by whoever needs it. Value and
// tag arrive together, so there is nothing to order and no fence; a word is written once
// a layer, by one thread. Its next value is stored only after all of its readers are
// done, because each phase needs all words of the one before (q/k/v: the heads' own, all
// heads together all), through all five phases of a layer. The words are cleared (tag 0,
// no layer's) by a launch before.
//
// No wait is without end: tiles are numbered in the order of their phases, a tile waits
// for lower numbers only, and a workgroup takes the next number when it runs (an atomic
// counter). So the lowest unfinished tile always has what it waits for, whatever part of
// the grid is resident and whatever else runs on the device.
//
// A step of 24 layers of 896 (14 heads over 2 x 64, 4,864 gated, head of 151,936), us, a
// launch a phase / here: one request of 600 740 / 445, of 16,000 957 / 745; two of 600
// 780 / 515; four of 600 885 / 680, of 4,000 973 / 884. The layers alone: 385 for one of
// 600, 330 where no weights are read: looks stand behind others' weights in a CU's
// queue, which is why a wave has one load of W underway at a time (all of them: 418).
// Tried: all waves looking at all they need until it is there 480 (each sleeps until one
// word of it is there, and before that until one of the phase before); operands out of
// the words without LDS 394; every word in two to eight copies 378.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "decode_common.h"

#define INL __attribute__((always_inline))

#define DS_LAYERS 32       // a launch
#define DS_THREADS 512
#define DS_WAVES 8
#define DS_UNIT 256        // tokens of a sequence that a workgroup takes at a time
#define DS_MAX_PARTS 8     // of the sequences together
#define DS_MAX_HEADS 1024  // values of all query heads, 64 or 128 each
// words of the attention's parts in LDS: of a part D + 2 a head
#define DS_STAGE (DS_MAX_PARTS * (DS_MAX_HEADS + DS_MAX_HEADS / 64 * 2))

struct StackLayer {
  const uint16_t *norm1, *w_qkv, *b_qkv, *w_o, *norm2, *w_gu, *w_d;
  uint16_t *k_cache, *v_cache;
};

struct StackArgs {
  StackLayer layer[DS_LAYERS];
  const uint16_t* x;          // [M, H]
  uint16_t *x_out, *res_out;  // [M, H] of the last layer
  unsigned long long* words;
  uint32_t* ticket;
  const int *positions, *seq_lens, *block_tables;
  const int64_t* slots;
  const float* cos_sin;       // [.., D]
  int M, H, Hq, Hk, F, G, layers, first, all;  // first: layers of launches before
  int max_blocks, bs_shift, parts;
  int n1, n2, n3, n4, n5;     // workgroups of the phases
  int at_att, at_v3, at_act, at_v5;  // words; q/k/v at 0
  float eps, scale;
};

namespace {

typedef unsigned long long u64;
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

DEVINL void put(u64* p, uint32_t v, uint32_t tag) {
  __hip_atomic_store(p, ((u64)tag << 32) | v, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

DEVINL u64 look(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the first n words at `at`, as soon as all of them carry the tag
template <int N>
DEVINL void take(const u64* words, const uint32_t (&at)[N], uint32_t tag,
                 uint32_t (&v)[N], int n = N) {
  for (;;) {
    u64 w[N];
    bool ok = true;
#pragma unroll
    for (int i = 0; i < N; ++i)  // 32 bits beside one base
      if (i < n)
        w[i] = look(reinterpret_cast<const u64*>(
            reinterpret_cast<const uint8_t*>(words) + (size_t)(at[i] * 8)));
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if (i >= n) break;
      ok = ok && (uint32_t)(w[i] >> 32) == tag;
      v[i] = (uint32_t)w[i];
    }
    if (ok) break;
    __builtin_amdgcn_s_sleep(1);
  }
}

// Until a word is there. Whoever is far ahead looks rarely, and at one word, or the
// words' memory is busy with looks.
template <int SLEEP>
DEVINL void until(const u64* word, uint32_t tag) {
  for (;;) {
    if ((uint32_t)(look(word) >> 32) == tag) break;
    __builtin_amdgcn_s_sleep(SLEEP);
  }
}

// s_barrier behind this wave's LDS accesses; loads from memory stay in flight
DEVINL void meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

DEVINL float lo16(uint32_t v) { return __uint_as_float(v << 16); }
DEVINL float hi16(uint32_t v) { return __uint_as_float(v & 0xffff0000u); }
DEVINL uint32_t pack(float a, float b) {
  return f32_to_bf16_bits(a) | ((uint32_t)f32_to_bf16_bits(b) << 16);
}
DEVINL float rounded(float v) { return bf16_bits_to_f32(f32_to_bf16_bits(v)); }
DEVINL float silu(float g) { return g / (1.f + __expf(-g)); }

template <int V> using Int = std::integral_constant<int, V>;

}  // namespace

// A value of another lane of a row of 16: lane i has that of lane i + N.
template <int N>
DEVINL u32x4v from(u32x4v v) {
  if constexpr (N == 0) return v;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    v[i] = __builtin_amdgcn_update_dpp(0, v[i], 0x120 + (16 - N), 0xf, 0xf, false);
  return v;
}

template <int CTRL>
DEVINL float moved(float v) {
  return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), CTRL, 0xf,
                                                     0xf, false));
}
// the sum over 8 neighbouring lanes, and over all: a tenth of the time of shuffles
DEVINL float sum8(float v) {
  v += moved<0xb1>(v);   // lanes 1, 0, 3, 2
  v += moved<0x4e>(v);   // lanes 2, 3, 0, 1
  return v + moved<0x141>(v);  // half rows mirrored
}
DEVINL float sum64(float v) {
  v = sum8(v);
  v += moved<0x140>(v);  // rows mirrored
  return over_head(v, [](float a, float b) { return a + b; });
}

// One phase's product: tiles of 16 rows of W (gated: 8 of each half), KW waves share the
// at most S KW steps of 32 along K, R tiles each; all of W is here before the input is.
//
// The input is the second operand, of whose 16 columns only the first MB are rows of X.
// So a lane holds those of 16 / MB steps, read at once, and a step's come to the first
// columns by a turn of each 16 lanes.
template <int S, int KW, int R, int MB>
struct Product {
  static constexpr int PER = 16 / MB;               // steps a set of operands
  static constexpr int SETS = (S + PER - 1) / PER;
  bf16x8v w[R][S];
  u32x4v x[SETS];
  int begin, mine;  // this wave's steps

  DEVINL void start(const uint16_t* weight, int K, int tile0, int tiles, bool gated,
                    int half) {
    const int lane = threadIdx.x & 63, l15 = lane & 15, l4 = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int steps = K / 32, per = (steps + KW - 1) / KW;
    begin = min((wid % KW) * per, steps - 1);
    mine = max(0, min(per, steps - (wid % KW) * per));
    const uint16_t* row[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int tile = min(tile0 + (wid / KW) * R + r, tiles - 1);
      const int n = gated ? tile * 8 + (l15 & 7) + (l15 < 8 ? 0 : half) : tile * 16 + l15;
      row[r] = weight + (size_t)n * K + begin * 32 + l4 * 8;
    }
    // past its steps a wave asks for its last one again: no branch among the loads
#pragma unroll
    for (int s = 0; s < S; ++s) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        w[r][s] = *reinterpret_cast<const bf16x8v*>(row[r] + max(0, min(s, mine - 1)) * 32);
#pragma unroll
      for (int r = 0; r < R; ++r) asm volatile("" : "+v"(w[r][s]));  // here by now
    }
  }

  // where along K, and in which row, the eight values of this lane in set i are
  DEVINL int at(int i) const {
    const int step = i * PER + (int)(threadIdx.x & 15) / MB;
    return (begin + max(0, min(step, mine - 1))) * 32 + (threadIdx.x >> 4 & 3) * 8;
  }
  static DEVINL int x_row(int M) { return min((int)(threadIdx.x % MB), M - 1); }

  // part: [wave][R][MB][16]
  DEVINL void run(float* part, int M) {
    const int lane = threadIdx.x & 63, l15 = lane & 15, l4 = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    f32x4v acc[R] = {};
    each<0>(acc);
    if (l15 < M)
#pragma unroll
      for (int r = 0; r < R; ++r)
        *reinterpret_cast<f32x4v*>(part + ((wid * R + r) * MB + l15) * 16 + l4 * 4) =
            acc[r];
  }

  template <int s>
  DEVINL void each(f32x4v (&acc)[R]) {
    if constexpr (s < S) {
      if (s < mine) {
        const bf16x8v xf =
            __builtin_bit_cast(bf16x8v, from<s % PER * MB>(x[s / PER]));
#pragma unroll
        for (int r = 0; r < R; ++r)
          acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[r][s], xf, acc[r], 0, 0, 0);
      }
      each<s + 1>(acc);
    }
  }

  // the sum of result n of row m of local tile t
  static DEVINL float sum(const float* part, int t, int m, int n) {
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < KW; ++k)
      v += part[(((t / R * KW + k) * R + t % R) * MB + m) * 16 + n];
    return v;
  }
};

template <int D, int MB>
__global__ __launch_bounds__(DS_THREADS, 4) void decode_stack_kernel(const StackArgs p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  // of the products: the waves' sums, then their input
  float* const part = reinterpret_cast<float*>(smem);
  uint32_t* const in = reinterpret_cast<uint32_t*>(smem + DS_WAVES * 2 * 4 * 16 * 4);
  __shared__ uint32_t ticket;
  __shared__ float ssq[DS_WAVES][MB];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l4 = lane >> 4;
  if (tid == 0)
    ticket = __hip_atomic_fetch_add(p.ticket, 1u, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const int per_layer = p.n1 + p.n2 + p.n3 + p.n4 + p.n5;
  const int t = __builtin_amdgcn_readfirstlane(ticket);
  const int li = t / per_layer;
  if (li >= p.layers) return;
  int wg = t - li * per_layer;
  const StackLayer& L = p.layer[li];
  const uint32_t tag = p.first + li + 1;  // this layer's
  const bool initial = p.first + li == 0;
  u64* const words = p.words;
  const int M = p.M, H = p.H;

  using Qkv = Product<8, 4, 1, MB>;
  using Out = Product<4, 8, 1, MB>;
  using Gated = Product<8, 4, 2, MB>;
  using Down = Product<20, 8, 1, MB>;

  // the first wave's lanes: pair of neighbouring results, row, tile
  const int pr = lane & 7, pm = (lane >> 3) % M, pt = (lane >> 3) / M;

  // n words to LDS, of at(i) to dst[i]; a barrier is the caller's
  auto collect = [&](int n, uint32_t* dst, uint32_t tg, auto at) INL {
    constexpr int NB = 6;
    for (int j0 = 0; j0 < n; j0 += NB * DS_THREADS) {
      uint32_t a[NB], w[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i) a[i] = at(min(j0 + i * DS_THREADS + tid, n - 1));
      take(words, a, tg, w, min(NB, (n - j0 + DS_THREADS - 1) / DS_THREADS));
#pragma unroll
      for (int i = 0; i < NB; ++i)
        if (j0 + i * DS_THREADS + tid < n) dst[j0 + i * DS_THREADS + tid] = w[i];
    }
  };

  // The product with the residual stream times the norm's gain. 1 / rms is a factor of
  // the results, returned, of row `of`, to the first wave. v: the stream's words, then
  // those of its squares' sums; tg 0: the stack's input. late: a word of the awaited
  // phase, early: of the one before.
  auto normed = [&](auto& prod, const uint16_t* gain, int v, uint32_t tg, int of,
                    const u64* early, const u64* late) INL {
    using P = std::remove_reference_t<decltype(prod)>;
    constexpr int SETS = P::SETS;
    const int pairs = H / 2, sums = H / 16, m = P::x_row(M);
    bf16x8v g[SETS];
#pragma unroll
    for (int i = 0; i < SETS; ++i)
      g[i] = *reinterpret_cast<const bf16x8v*>(gain + prod.at(i));
#pragma unroll
    for (int i = 0; i < SETS; ++i) asm volatile("" : "+v"(g[i]));
    float ss[MB] = {};
    if (tg == 0) {
#pragma unroll
      for (int n = 0; n < MB; ++n)
        if (n < M) {
          const uint32_t* x = reinterpret_cast<const uint32_t*>(p.x + (size_t)n * H);
          for (int j = tid; j < pairs; j += DS_THREADS) {
            const uint32_t w = x[j];
            const float a = lo16(w), b = hi16(w);
            ss[n] += a * a + b * b;
            in[n * pairs + j] = w;
          }
          ss[n] = sum64(ss[n]);
          if (lane == 0) ssq[wid][n] = ss[n];
        }
    } else {
      if (wid == 0) {
        until<16>(early, tg);
        until<4>(late, tg);
      }
      meet();
      collect(M * (pairs + sums), in, tg, [&](int i) INL { return (uint32_t)(v + i); });
    }
    meet();
#pragma unroll
    for (int i = 0; i < SETS; ++i) {
      const u32x4v w = *reinterpret_cast<const u32x4v*>(in + m * pairs + prod.at(i) / 2);
      const u32x4v gw = __builtin_bit_cast(u32x4v, g[i]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        prod.x[i][j] = pack_bf16(lo16(w[j]) * lo16(gw[j]), hi16(w[j]) * hi16(gw[j]));
    }
    prod.run(part, M);
    if (wid == 0)
#pragma unroll
      for (int n = 0; n < MB; ++n) {
        if (n >= M) break;
        if (tg == 0) {
          ss[n] = lane < DS_WAVES ? ssq[lane][n] : 0.f;
        } else {
          ss[n] = lane < sums ? __uint_as_float(in[M * pairs + n * sums + lane]) : 0.f;
        }
        ss[n] = sum64(ss[n]);
      }
    meet();
    float mine = ss[0];
#pragma unroll
    for (int n = 1; n < MB; ++n) mine = of == n ? ss[n] : mine;
    return rsqrtf(mine / H + p.eps);
  };

  if (wg < p.n1) {  // ---- norm, q/k/v ------------------------------------------------------
    const int N = (p.Hq + 2 * p.Hk) * D, tiles = N / 16, tile0 = wg * 2;
    Qkv prod;
    prod.start(L.w_qkv, H, tile0, tiles, false, 0);
    const bool mine = wid == 0 && pt < 2 && tile0 + pt < tiles;
    float b0 = 0.f, b1 = 0.f;
    if (mine && L.b_qkv != nullptr) {
      const int n = (tile0 + pt) * 16 + pr * 2;
      b0 = bf16_bits_to_f32(L.b_qkv[n]);
      b1 = bf16_bits_to_f32(L.b_qkv[n + 1]);
    }
    const float rstd = normed(prod, L.norm1, p.at_v5, tag - 1, pm,
                              words + p.at_act + wg * 37 % (p.F / 2),
                              words + p.at_v5 + wg * 11 % (H / 2));
    if (mine)
      put(words + (size_t)pm * (N / 2) + (tile0 + pt) * 8 + pr,
          pack(Qkv::sum(part, pt, pm, pr * 2) * rstd + b0,
               Qkv::sum(part, pt, pm, pr * 2 + 1) * rstd + b1), tag);
    return;
  }
  wg -= p.n1;

  if (wg < p.n2) {  // ---- rope, cache, attention: a row, a head, a part ---------------------
    constexpr int KC = D / 32, MT = D / 16, MROW = D + 4;
    const int piece = wg % p.parts, hk = wg / p.parts % p.Hk, m = wg / p.parts / p.Hk;
    const int G = p.G, len = p.seq_lens[m];
    const int units = (len + DS_UNIT - 1) / DS_UNIT;
    if (piece >= max(1, min(p.parts, units))) return;
    const int pos = p.positions[m];
    const int64_t slot = p.slots[m];
    const int BS = 1 << p.bs_shift;
    // [16][D + 8]: heads, then the new key
    uint16_t* const qs = reinterpret_cast<uint16_t*>(smem);
    uint16_t* const vn = qs + 16 * (D + 8);    // [D] the new value
    float* const ms = reinterpret_cast<float*>(vn + D);  // [waves][16]
    float* const ls = ms + DS_WAVES * 16;
    float* const sums = ls + DS_WAVES * 16;    // [waves][G][MROW]
    const auto* btab = (const __attribute__((address_space(4))) int*)(
        p.block_tables + (size_t)m * p.max_blocks);
    const int last = (len - 1) & ~31;
    const int rr = 8 * (l15 >> 2) + (l15 & 3);

    bf16x8v kr[2][KC], vr[MT];
    auto load = [&](int tok) INL {
      const int64_t page_elems = (int64_t)p.Hk << p.bs_shift;
      const int p0 = btab[tok >> p.bs_shift];
      const int p1 = btab[min(p.bs_shift == 4 ? tok + 16 : tok, len - 1) >> p.bs_shift];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int k = rr + 4 * t;
        const int64_t page = p.bs_shift == 4 && k >= 16 ? p1 : p0;
        const uint16_t* src = L.k_cache +
            (page * page_elems + hk * BS + ((tok + k) & (BS - 1))) * D + l4 * 8;
#pragma unroll
        for (int s = 0; s < KC; ++s)
          kr[t][s] = *reinterpret_cast<const bf16x8v*>(src + s * 32);
      }
      const int64_t page = p.bs_shift == 4 && l4 >= 2 ? p1 : p0;
      const uint16_t* src = L.v_cache + (page * page_elems + hk * BS) * D + l15 * BS +
                            ((tok + l4 * 8) & (BS - 1));
#pragma unroll
      for (int d = 0; d < MT; ++d)
        vr[d] = *reinterpret_cast<const bf16x8v*>(src + d * 16 * BS);
    };
    int tok = piece * DS_UNIT + wid * 32;
    const int hop = p.parts * DS_UNIT;
    if (tok < len) load(tok);

    // a thread turns two neighbouring pairs of one head (or of the key)
    const int th = tid / (D / 4), tj = tid % (D / 4);
    f32x2v cs = {}, sn = {};
    if (th <= G) {
      cs = *reinterpret_cast<const f32x2v*>(p.cos_sin + (size_t)pos * D + tj * 2);
      sn = *reinterpret_cast<const f32x2v*>(p.cos_sin + (size_t)pos * D + D / 2 + tj * 2);
    }
    if (!initial) {
      if (wid == 0) until<16>(words + p.at_v5 + wg * 11 % (H / 2), tag - 1);
      meet();
    }
    {
      const int row = m * ((p.Hq + 2 * p.Hk) * D / 2);
      const int head = min(th, G) < G ? hk * G + min(th, G) : p.Hq + hk;
      uint32_t at[3], w[3];
      at[0] = row + head * (D / 2) + tj;
      at[1] = at[0] + D / 4;
      at[2] = row + (p.Hq + p.Hk + hk) * (D / 2) + tid % (D / 2);
      take(words, at, tag, w);
      if (th <= G) {
        const float x0 = lo16(w[0]), x1 = hi16(w[0]), y0 = lo16(w[1]), y1 = hi16(w[1]);
        uint32_t* dst = reinterpret_cast<uint32_t*>(qs + th * (D + 8)) + tj;
        const uint32_t a = pack_bf16(fmaf(x0, cs[0], -y0 * sn[0]),
                                     fmaf(x1, cs[1], -y1 * sn[1]));
        const uint32_t b = pack_bf16(fmaf(y0, cs[0], x0 * sn[0]),
                                     fmaf(y1, cs[1], x1 * sn[1]));
        dst[0] = a;
        dst[D / 4] = b;
      }
      if (tid < D / 2) reinterpret_cast<uint32_t*>(vn)[tid] = w[2];
    }
    meet();
    // where this workgroup's unit holds the new token: into the cache
    const bool fresh = slot >= 0 && units > 0 && (units - 1) % p.parts == piece;
    const int r = (len - 1) & 31;
    if (fresh) {
      const int64_t row = (slot >> p.bs_shift) * p.Hk + hk;
      const int in = (int)(slot & (BS - 1));
      if (tid < D / 8)
        *reinterpret_cast<bf16x8v*>(L.k_cache + (row * BS + in) * D + tid * 8) =
            *reinterpret_cast<const bf16x8v*>(qs + G * (D + 8) + tid * 8);
      else if (tid >= 64 && tid < 64 + D)
        L.v_cache[(row * D + tid - 64) * BS + in] = vn[tid - 64];
    }
    bf16x8v qf[KC];
#pragma unroll
    for (int s = 0; s < KC; ++s)
      qf[s] = *reinterpret_cast<const bf16x8v*>(qs + min(l15, G - 1) * (D + 8) + s * 32 +
                                                l4 * 8);
    f32x4v o[MT] = {};
    float mx_ = -1e30f, l = 0.f;
    const float c = p.scale * 1.4426950408889634f;
    for (; tok < len; tok += hop) {
      if (fresh && tok == last) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
          if (rr + 4 * t == r)
#pragma unroll
            for (int s = 0; s < KC; ++s)
              kr[t][s] = *reinterpret_cast<const bf16x8v*>(qs + G * (D + 8) + s * 32 +
                                                           l4 * 8);
        if (l4 == r >> 3)
#pragma unroll
          for (int d = 0; d < MT; ++d) {
            u32x4v a = __builtin_bit_cast(u32x4v, vr[d]);
            const uint32_t n = vn[d * 16 + l15];
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (i == (r & 7) >> 1)
                a[i] = r & 1 ? (a[i] & 0xffffu) | n << 16 : (a[i] & 0xffff0000u) | n;
            vr[d] = __builtin_bit_cast(bf16x8v, a);
          }
      }
      // token of s[t][r]: tok + 8 l4 + 4 t + r
      f32x4v s[2] = {};
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int k = 0; k < KC; ++k)
          s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kr[t][k], qf[k], s[t], 0, 0, 0);
      const bool cut = tok + 32 > len;
      if (cut)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          s[e >> 2][e & 3] =
              tok + 8 * l4 + e < len ? s[e >> 2][e & 3] : -__builtin_inff();
      float mx = s[0][0];
#pragma unroll
      for (int e = 1; e < 8; ++e) mx = fmaxf(mx, s[e >> 2][e & 3]);
      mx = over_head(mx, [](float a, float b) { return fmaxf(a, b); }) * c;
      const float m2 = fmaxf(mx_, mx);
      const float f = __builtin_amdgcn_exp2f(mx_ - m2);
      mx_ = m2;
      l *= f;
#pragma unroll
      for (int d = 0; d < MT; ++d) o[d] *= f;
      u32x4v pk;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float q0 = __builtin_amdgcn_exp2f(fmaf(s[e >> 2][e & 3], c, -mx_));
        const float q1 = __builtin_amdgcn_exp2f(fmaf(s[e >> 2][(e & 3) + 1], c, -mx_));
        l += q0 + q1;
        pk[e >> 1] = pack_bf16(q0, q1);
      }
      // slots past the end may hold anything: weight 0 times it
      if (cut) {
        const int n = len - tok - 8 * l4;
        u32x4v keep;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          keep[i] = n >= 2 * i + 2 ? ~0u : n == 2 * i + 1 ? 0xffffu : 0u;
#pragma unroll
        for (int d = 0; d < MT; ++d)
          vr[d] = __builtin_bit_cast(bf16x8v, __builtin_bit_cast(u32x4v, vr[d]) & keep);
      }
      const bf16x8v pb = __builtin_bit_cast(bf16x8v, pk);
#pragma unroll
      for (int d = 0; d < MT; ++d)
        o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vr[d], pb, o[d], 0, 0, 0);
      if (tok + hop < len) load(tok + hop);
    }
    l = over_head(l, [](float a, float b) { return a + b; });
    if (l4 == 0) {
      ms[wid * 16 + l15] = mx_;
      ls[wid * 16 + l15] = l;
    }
    if (l15 < G)
#pragma unroll
      for (int d = 0; d < MT; ++d)
        *reinterpret_cast<f32x4v*>(sums + (wid * G + l15) * MROW + d * 16 + l4 * 4) = o[d];
    meet();
    for (int e = tid; e < G * D; e += DS_THREADS) {
      const int g = e / D, d = e % D;
      float mg = -1e30f, lg = 0.f, v = 0.f;
#pragma unroll
      for (int w = 0; w < DS_WAVES; ++w) mg = fmaxf(mg, ms[w * 16 + g]);
#pragma unroll
      for (int w = 0; w < DS_WAVES; ++w) {
        const float f = __builtin_amdgcn_exp2f(ms[w * 16 + g] - mg);
        lg = fmaf(ls[w * 16 + g], f, lg);
        v = fmaf(sums[(w * G + g) * MROW + d], f, v);
      }
      u64* const to = words + p.at_att + (m * p.parts + piece) * (p.Hq * (D + 2)) +
                      (hk * G + g) * (D + 2);
      put(to + d, __float_as_uint(v), tag);
      if (d < 2) put(to + D + d, __float_as_uint(d ? lg : mg), tag);
    }
    return;
  }
  wg -= p.n2;

  // a projection's results: the residual stream then, and its squares' sums
  auto publish = [&](int tile, int m, int q, float a, float b, uint32_t old, int v,
                     bool out) INL {
    const float a0 = rounded(a), b0 = rounded(b);
    if (out) {
      const size_t at = (size_t)m * (H / 2) + tile * 8 + q;
      reinterpret_cast<uint32_t*>(p.x_out)[at] = pack(a, b);
      reinterpret_cast<uint32_t*>(p.res_out)[at] = old;
      return;
    }
    const float a1 = a0 + lo16(old), b1 = b0 + hi16(old);
    put(words + v + m * (H / 2) + tile * 8 + q, pack(a1, b1), tag);
    const float ss = sum8(a1 * a1 + b1 * b1);
    if (q == 0)
      put(words + v + M * (H / 2) + m * (H / 16) + tile, __float_as_uint(ss), tag);
  };

  if (wg < p.n3) {  // ---- the parts of the attention, output product ---------------------
    const int K = p.Hq * D, tiles = H / 16;
    Out prod;
    prod.start(L.w_o, K, wg, tiles, false, 0);
    if (wid == 0) until<16>(words + wg * 11 % ((p.Hq + 2 * p.Hk) * D / 2), tag);
    const bool mine = wid == 0 && pt < 1;
    uint32_t old = 0;
    if (mine) {
      const int at = pm * (H / 2) + wg * 8 + pr;
      if (initial) {
        old = reinterpret_cast<const uint32_t*>(p.x)[at];
      } else {
        uint32_t a[1] = {(uint32_t)(p.at_v5 + at)}, w[1];
        take(words, a, tag - 1, w);
        old = w[0];
      }
    }
    if (wid == 0) until<4>(words + p.at_att + wg * 37 % (p.Hq * D), tag);
    meet();
    constexpr int W = D + 2;
    uint32_t* const xs = in + DS_STAGE;
    int begin[MB + 1];  // of the rows' parts in LDS
    begin[0] = 0;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      int words = 0;
      if (m < M) {
        const int units = (p.seq_lens[m] + DS_UNIT - 1) / DS_UNIT;
        words = max(1, min(p.parts, units)) * p.Hq * W;
      }
      begin[m + 1] = begin[m] + words;
    }
    collect(begin[MB], in, tag, [&](int i) INL {
      int row = 0, from = 0;
#pragma unroll
      for (int q = 1; q < MB; ++q)
        if (i >= begin[q] && q < M) row = q, from = begin[q];
      return (uint32_t)(p.at_att + row * p.parts * p.Hq * W + i - from);
    });
    meet();
    for (int j = tid; j < M * (K / 2); j += DS_THREADS) {
      const int row = j / (K / 2), k = j % (K / 2) * 2;
      int from = 0, to = begin[1];
#pragma unroll
      for (int q = 1; q < MB; ++q)
        if (row == q) from = begin[q], to = begin[q + 1];
      const float* src = reinterpret_cast<const float*>(in) + k / D * W;
      float mall = -1e30f, l = 0.f, a = 0.f, b = 0.f;
      for (int o = from; o < to; o += p.Hq * W) mall = fmaxf(mall, src[o + D]);
      for (int o = from; o < to; o += p.Hq * W) {
        const float g = __builtin_amdgcn_exp2f(src[o + D] - mall);
        l += src[o + D + 1] * g;
        a += src[o + k % D] * g;
        b += src[o + k % D + 1] * g;
      }
      const float inv = l > 0.f ? 1.f / l : 0.f;  // no tokens: zeros
      xs[row * (K / 2) + k / 2] = pack_bf16(a * inv, b * inv);
    }
    meet();
    prod.x[0] = *reinterpret_cast<const u32x4v*>(xs + Out::x_row(M) * (K / 2) +
                                                 prod.at(0) / 2);
    prod.run(part, M);
    meet();
    if (mine)
      publish(wg, pm, pr, Out::sum(part, 0, pm, pr * 2),
              Out::sum(part, 0, pm, pr * 2 + 1), old, p.at_v3, false);
    return;
  }
  wg -= p.n3;

  if (wg < p.n4) {  // ---- norm, gate and up, silu ----------------------------------------
    const int tiles = p.F / 8, tile0 = wg * 4;
    Gated prod;
    prod.start(L.w_gu, H, tile0, tiles, true, p.F);
    const int q = lane & 3, m = (lane >> 2) % M, tt = (lane >> 2) / M;
    const float rstd = normed(prod, L.norm2, p.at_v3, tag, m,
                              words + p.at_att + wg * 37 % (p.Hq * D),
                              words + p.at_v3 + wg * 11 % (H / 2));
    if (wid == 0 && tt < 4 && tile0 + tt < tiles) {
      float y[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        y[i] = silu(rounded(Gated::sum(part, tt, m, q * 2 + i) * rstd)) *
               rounded(Gated::sum(part, tt, m, q * 2 + i + 8) * rstd);
      put(words + p.at_act + m * (p.F / 2) + (tile0 + tt) * 4 + q,
          pack(y[0], y[1]), tag);
    }
    return;
  }
  wg -= p.n4;

  {  // ---- down product --------------------------------------------------------------------
    const int tiles = H / 16, pairs = p.F / 2;
    Down prod;
    prod.start(L.w_d, p.F, wg, tiles, false, 0);
    if (wid == 0) until<16>(words + p.at_v3 + wg * 11 % (H / 2), tag);
    const bool mine = wid == 0 && pt < 1;
    uint32_t old = 0;
    if (mine) {
      uint32_t a[1] = {(uint32_t)(p.at_v3 + pm * (H / 2) + wg * 8 + pr)}, w[1];
      take(words, a, tag, w);
      old = w[0];
    }
    if (wid == 0) until<4>(words + p.at_act + wg * 37 % (p.F / 2), tag);
    meet();
    collect(M * pairs, in, tag, [&](int i) INL { return (uint32_t)(p.at_act + i); });
    meet();
#pragma unroll
    for (int i = 0; i < Down::SETS; ++i)
      prod.x[i] = *reinterpret_cast<const u32x4v*>(in + Down::x_row(M) * pairs +
                                                   prod.at(i) / 2);
    prod.run(part, M);
    meet();
    if (mine)
      publish(wg, pm, pr, Down::sum(part, 0, pm, pr * 2),
              Down::sum(part, 0, pm, pr * 2 + 1), old, p.at_v5,
              p.first + li == p.all - 1);
  }
}

__global__ void decode_stack_clear_kernel(unsigned long long* words, int n,
                                          uint32_t* tickets, int launches) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) words[i] = 0;
  if (i < launches) tickets[i * 32] = 0;
}

struct StackSizes {
  int M, H, Hq, Hk, D, F, max_len;
};

namespace {

int stack_parts(const StackSizes& s) {
  return clamp_int(ceil_div(s.max_len, DS_UNIT), 1, DS_MAX_PARTS / s.M);
}

int stack_lds(const StackSizes& s) {
  // the waves' sums; the stream, the parts and their sum, or the gated product
  const int room = std::max({s.M * (s.H / 2 + s.H / 16),
                             DS_STAGE + s.M * s.Hq * s.D / 2, s.M * s.F / 2});
  const int product = DS_WAVES * 2 * 4 * 16 * 4 + room * 4;
  const int G = s.Hq / s.Hk;
  const int attention = 16 * (s.D + 8) * 2 + s.D * 2 + 2 * DS_WAVES * 16 * 4 +
                        DS_WAVES * G * (s.D + 4) * 4;
  return std::max(product, attention);
}

}  // namespace

// Widths whose products a workgroup's registers hold, and contexts up to eight units of 64
// values, four of 128, a part: a workgroup takes its units one after the other, 64 KB of K
// and V each, where launches apart deal them to the whole chip. Over 460 sizes drawn at
// random, stacks of eight layers and more so many times as fast as launches apart, in the
// mean and all: units x D to 256 1.54 (1.12 .. 1.94), to 384 1.21 (1.07 .. 1.39), to 512
// 1.10 (0.93 .. 1.29), to 640 0.87 (0.81 .. 0.94), above 0.70. The two launches' start, some
// 10 us, is a part of every call: one layer 1.09 (0.86 .. 1.28) to 256, two 1.19 (0.94 ..).
extern "C" bool decode_stack_takes(const StackSizes* s) {
  if (s->M < 1 || s->M > 4 || s->Hk < 1 || s->Hq % s->Hk || s->Hq / s->Hk > 15) return false;
  if (s->D != 64 && s->D != 128) return false;
  if (s->H % 32 || s->H < 32 || s->H > 1024 || s->Hq * s->D > DS_MAX_HEADS) return false;
  if (s->F % 32 || s->F < 32 || s->F > 5120) return false;
  return s->max_len >= 1 &&
         ceil_div(ceil_div(s->max_len, DS_UNIT), stack_parts(*s)) * s->D <= 512;
}

// 64-bit words of the workspace before the counters, 32 words a launch; at: see StackArgs
extern "C" int64_t decode_stack_words(const StackSizes* s, int (*at)[4]) {
  const int parts = stack_parts(*s);
  int64_t n = (int64_t)s->M * (s->Hq + 2 * s->Hk) * s->D / 2;
  const int64_t stream = (int64_t)s->M * (s->H / 2 + s->H / 16);
  const int64_t size[4] = {(int64_t)s->M * parts * s->Hq * (s->D + 2), stream,
                           (int64_t)s->M * s->F / 2, stream};
  for (int i = 0; i < 4; ++i) {
    n = (n + 15) / 16 * 16;
    if (at != nullptr) (*at)[i] = (int)n;
    n += size[i];
  }
  return n;
}

extern "C" void launch_decode_stack(
    const StackSizes* s, const void* const* pointers, int layers, const void* x,
    void* x_out, void* res_out, void* work, const int* positions, const int* seq_lens,
    const int* block_tables, const int64_t* slots, const float* cos_sin, int max_blocks,
    int bs_shift, float eps, float scale, hipStream_t stream) {
  int at[4];
  const int64_t n = decode_stack_words(s, &at);
  const int launches = ceil_div(layers, DS_LAYERS);
  u64* words = (u64*)work;
  uint32_t* tickets = (uint32_t*)(words + n);
  decode_stack_clear_kernel<<<ceil_div((int)n, 256), 256, 0, stream>>>(words, (int)n,
                                                                      tickets, launches);
  const int lds = stack_lds(*s);
  StackArgs p{};
  p.x = (const uint16_t*)x;
  p.x_out = (uint16_t*)x_out;
  p.res_out = (uint16_t*)res_out;
  p.words = words;
  p.positions = positions;
  p.seq_lens = seq_lens;
  p.block_tables = block_tables;
  p.slots = slots;
  p.cos_sin = cos_sin;
  p.M = s->M;
  p.H = s->H;
  p.Hq = s->Hq;
  p.Hk = s->Hk;
  p.F = s->F;
  p.G = s->Hq / s->Hk;
  p.all = layers;
  p.max_blocks = max_blocks;
  p.bs_shift = bs_shift;
  p.parts = stack_parts(*s);
  p.n1 = ceil_div((s->Hq + 2 * s->Hk) * s->D / 16, 2);
  p.n2 = s->M * s->Hk * p.parts;
  p.n3 = s->H / 16;
  p.n4 = ceil_div(s->F / 8, 4);
  p.n5 = s->H / 16;
  p.at_att = at[0];
  p.at_v3 = at[1];
  p.at_act = at[2];
  p.at_v5 = at[3];
  p.eps = eps;
  p.scale = scale;
  for (int l = 0; l < launches; ++l) {
    p.first = l * DS_LAYERS;
    p.layers = layers - p.first < DS_LAYERS ? layers - p.first : DS_LAYERS;
    p.ticket = tickets + l * 32;
    for (int i = 0; i < p.layers; ++i) {
      const void* const* q = pointers + (size_t)(p.first + i) * 9;
      p.layer[i] = {(const uint16_t*)q[0], (const uint16_t*)q[1], (const uint16_t*)q[2],
                    (const uint16_t*)q[3], (const uint16_t*)q[4], (const uint16_t*)q[5],
                    (const uint16_t*)q[6], (uint16_t*)q[7], (uint16_t*)q[8]};
    }
    const int grid = p.layers * (p.n1 + p.n2 + p.n3 + p.n4 + p.n5);
    auto go = [&](auto d, auto mb) {
      constexpr int D = decltype(d)::value, MB = decltype(mb)::value;
      decode_stack_kernel<D, MB><<<grid, DS_THREADS, lds, stream>>>(p);
    };
    auto rows = [&](auto d) {
      if (s->M == 1) go(d, Int<1>{});
      else if (s->M == 2) go(d, Int<2>{});
      else go(d, Int<4>{});
    };
    if (s->D == 64) rows(Int<64>{});
    else rows(Int<128>{});
  }
}
