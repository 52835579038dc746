// MLA decode attention over the compressed latent cache for gfx950.
//
//   S^T[64 tok x 16 heads] = C . Q^T     C = [latent | rope] rows, 576 values
//   O^T[512 x 16 heads]   += C_v^T . P   C_v = the latent part of the same rows
// All query heads share ONE cache row a token; a workgroup takes 64 heads, of whose Q and
// O^T its waves' registers hold all. With 128 heads two workgroups read a row, at the
// same time and through one XCD's L2. Both products read the one copy of a tile in LDS:
// S^T's operand rows are token rows; O^T's operand is transposed on the way out
// (ds_read_b64_tr_b16), and in the order in which the accumulators of S^T hold their
// tokens, so P stays in registers. 16-byte chunks are XOR-swizzled so that both kinds of
// read spread over the banks. An fp8 cache is widened on its way through registers.
//
// Every workgroup takes a run of tiles (find_run). Lengths are read on the device, so a
// captured step balances for any lengths. A sequence that lies in one run is finished
// there; the others leave fp32 parts that a second kernel adds up. Short sequences (256
// tokens at most) take a workgroup each and need no second kernel.
//
// Two kernels: mla_decode_wide_kernel for more than 32 heads on an fp8 cache,
// mla_decode_kernel for the others. What bounds them: with 64 heads the latent rows'
// stream, 4.0 us a CU for a tile of 64 tokens, 4.7 TB/s where a read alone reaches 6.1; with
// 128, whose two workgroups share a row in the L2, what a tile issues, 3.1 us; in fp8, 2.2
// and 1.8 us for 32 tokens, that too: 290 vector instructions and 34 products a wave that
// hardly overlap. And the start and end of a run, some 8 us of looking up, first rows and
// parts, then 9 of the second kernel.
//
// Reference analogue: parallax_extensions/kernels/mla/ (Metal, VALU); fresh
// MFMA design. Layout: cache [NB, BS, R+DR], q_latent [B, H, R], q_pe [B, H, DR].

#include <type_traits>

#include "common.h"
#include "mla_deal.h"

#define MLA_R 512
#define MLA_DR 64
#define MLA_DK 576          // values a cache row
#define MLA_ROW 1024        // bytes of a row's latent values in LDS
#define MLA_PE 128          // and of its rotated ones
#define MLA_KT 64           // tokens a tile,
#define MLA_DT 16           // 16-value tiles of O^T a wave
#define MLA_WT 32           // of the wide kernel
#define MLA_MIN_TOKENS 128  // a run is at least this long
#define MLA_MAX_RUNS 256    // one a CU

// the lambdas below are called once a buffer: left out of line, their captures
// would live in scratch
#define INL __attribute__((always_inline))

typedef short s16x4v __attribute__((ext_vector_type(4)));
typedef float f32x16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8n __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2n __attribute__((ext_vector_type(2)));

namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kHidden = -1e30f;

template <int V> using Int = std::integral_constant<int, V>;

DEVINL uint32_t pack_bf16(float a, float b) {
  bf16x2n p;
  p[0] = (__bf16)a;
  p[1] = (__bf16)b;
  return __builtin_bit_cast(uint32_t, p);
}

// 16 bytes a lane from memory to LDS, at + 16 lane, from a uniform base or a pointer a
// lane. In assembly: of the builtin the compiler knows that it writes LDS, and waits
// for copies in flight before reads of other places.
DEVINL void copy16(const uint8_t* base, uint32_t off, uint32_t at) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(off), "s"(base), "s"(at) : "m0", "memory");
}
DEVINL void copy16(const uint8_t* src, uint32_t at) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :: "v"(src), "s"(at) : "m0", "memory");
}

// over the four lanes that hold one head (l, l + 16, l + 32, l + 48)
template <class F>
DEVINL float over_head(float v, F f) {
  const auto a = __builtin_amdgcn_permlane16_swap(
      __float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// A tile in LDS: 64 rows of 64 chunks (the latent values), then 64 rows of 8 (the
// rotated ones). Chunk c of row r lies at c ^ row_xor(r), or rope_xor(r), which are
// linear over xor in the row's four bits. 16-byte reads go by lanes {0-3, 12-15,
// 20-23, 24-27} and so on, rows of one chunk and other rows of its neighbour, that is
// rows with bits 2 and 3 alike or not: they meet in no bank as no two such rows differ
// by 1 in row_xor. Transposing reads take two neighbouring chunks of 8 rows of one bit
// 3: those rows differ above bit 0.
DEVINL constexpr int row_xor(int r) { return (r & 7) * 2 ^ (r & 8 ? 9 : 0); }
DEVINL constexpr int rope_xor(int r) { return (r & 6) ^ (r & 8 ? 5 : 0); }

// tiles of sequence b: its tokens, or its list of token positions
template <bool SPARSE>
DEVINL int domain_of(const int* seq_lens, const int* topk, int max_topk,
                     int b) {
  if (SPARSE && topk[(size_t)b * max_topk] >= 0) return max_topk;
  return max(seq_lens[b], 0);
}

template <int CTRL>
DEVINL int moved(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false);
}
DEVINL int wave_sum(int v) {
  v += moved<0xb1>(v);   // lanes 1, 0, 3, 2
  v += moved<0x4e>(v);   // lanes 2, 3, 0, 1
  v += moved<0x141>(v);  // half rows mirrored
  v += moved<0x140>(v);  // rows mirrored
  return __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16) +
         __builtin_amdgcn_readlane(v, 32) + __builtin_amdgcn_readlane(v, 48);
}
DEVINL int sum_before(int v) {  // of lanes up to this one
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(v, o, WAVE_SIZE);
    if ((int)(threadIdx.x & 63) >= o) v += t;
  }
  return v;
}
// n / d rounded up, d > 0; exact to 2^21, and the same wherever it is asked
DEVINL int div_up(int n, int d) {
  return n > 0 ? (int)(((float)n - 0.5f) * __builtin_amdgcn_rcpf((float)d)) + 1 : 0;
}

// the first and the last run of each sequence, behind the parts' maxima and sums
DEVINL int2* part_runs(float* tmp_ml, int runs, int B, int H) {
  return reinterpret_cast<int2*>(tmp_ml + ((size_t)runs + B) * H * 2);
}

// How the tiles are dealt, found by one wave; tiles_of(b): of sequence b, 0 from B on.
// Each run lies in one sequence, which has as many of equal length as it takes for none
// to be longer than `per`, the least that `runs` suffice for. Or, where that is more than
// MORE tokens longer than even, runs go through the list of all tiles: a run that meets the
// next sequence pays the start and the end of a run twice, and leaves parts of both.
// What that is worth is measured by kernel and cache (us of a call, through the list / in
// one sequence, + how many tokens longer):
// - more than 32 heads, 384: 64 heads 24 x 5,158 +64 51.1 / 45.9, 238 of up to 1,077 +384
//   79 / 63; 128 heads 98 of up to 1,650 +320 66 / 54, 44 x 2,682 +384 70 / 73, 44 x 3,202 +512
//   77 / 84.
// - the same with an fp8 cache, in the wide kernel, 288: 128 heads 33 x 1,081 +96 46 / 42,
//   110 of up to 429 +288 50.9 / 42.2, 46 x 2,311 +320 74.8 / 80.4; 64 heads 93 x 2,749 +352
//   82.9 / 91.4.
// - up to 32 heads, 192: 16 heads 225 x 1,352 +128 84.4 / 77.0, 70 x 3,000 +192 49.2 / 46.3,
//   219 of up to 1,459 +448 48.4 / 55.9. fp8, 64: 165 of up to 1,388 +64 42.5 / 38.0, 107 of
//   up to 2,274 +128 48.0 / 53.1.
// - lists of 2,048 positions, more than 32 heads 192: 64 heads, 100 of them +192 91 / 86; 128
//   heads in fp8, 47 of them +256 82 / 87. Up to 32, 64: 40 of them +64 34.2 / 33.2, 100 of
//   them +192 64 / 68; in fp8 none longer: 40 of them +64 35 / 37.
template <int KT, int MORE, class F>
DEVINL Run find_run(int B, int run, int runs, F tiles_of) {
  const int lane = threadIdx.x & 63;
  // a lane's sequences: 256 in registers, as each pass would wait for their lengths again
  constexpr int KEPT = 4;
  int kept[KEPT] = {tiles_of(lane)};
  if (B > 64)
#pragma unroll
    for (int j = 1; j < KEPT; ++j) kept[j] = tiles_of(j * 64 + lane);
  auto each = [&](auto&& use) INL {
    use(kept[0]);
    if (B <= 64) return;
#pragma unroll
    for (int j = 1; j < KEPT; ++j) use(kept[j]);
    for (int b = KEPT * 64 + lane; b < B; b += 64) use(tiles_of(b));
  };
  int total = 0;
  each([&](int tiles) INL { total += tiles; });
  total = wave_sum(total);
  const int even = max(div_up(total, runs), MLA_MIN_TOKENS / KT);
  const int most = even + MORE / KT;
  const int least = least_length(even, most, runs, [&](int length) INL {
    int n = 0;
    each([&](int tiles) INL { n += div_up(tiles, length); });
    return wave_sum(n);
  });
  const bool whole = least <= most;
  const int per = whole ? least : even;
  const int begin = whole ? run : run * per;  // in runs, or in tiles
  int before = 0;
  for (int b0 = 0; b0 < B; b0 += 64) {
    int tiles = kept[0];
    if (b0 > 0) {
#pragma unroll
      for (int j = 1; j < KEPT; ++j) tiles = b0 == j * 64 ? kept[j] : tiles;
      if (b0 >= KEPT * 64) tiles = tiles_of(b0 + lane);
    }
    const int n = whole ? div_up(tiles, per) : tiles;
    const int sum = before + sum_before(n);
    const unsigned long long hit = __ballot(begin >= sum - n && begin < sum);
    if (hit) {
      const int src = __ffsll(hit) - 1;
      const int k = __builtin_amdgcn_readlane(n, src);
      const int first = __builtin_amdgcn_readlane(sum, src) - k;
      if (!whole) return run_of_list(b0 + src, begin, first, per, total);
      return run_of_sequence(b0 + src, run - first, __builtin_amdgcn_readlane(tiles, src), k,
                             div_up);
    }
    before = __builtin_amdgcn_readlane(sum, 63);
  }
  return {0, 0, 0, 1};
}

}  // namespace

template <int W, bool KV_FP8, bool SPARSE>
__global__ __launch_bounds__(W * 64, 2) void mla_decode_kernel(
    uint16_t* __restrict__ out,             // [B, H, R]
    float* __restrict__ tmp_acc,            // [parts, H, R]; null: a workgroup
    float* __restrict__ tmp_ml,             // [parts, H, 2]      a sequence
    const uint16_t* __restrict__ q_latent,  // [B, H, R]
    const uint16_t* __restrict__ q_pe,      // [B, H, DR]
    const void* __restrict__ cache,         // [NB, BS, R+DR] bf16 | fp8(e4m3)
    const int* __restrict__ block_tables,   // [B, max_blocks]
    const int* __restrict__ seq_lens,
    const int* __restrict__ topk,           // [B, max_topk] (SPARSE)
    const int max_topk, const int B, const int max_blocks, const int H,
    const int bs_shift, const float scale) {
  // see find_run
  constexpr int MORE =
      W == 8 ? (SPARSE ? 192 : 384) : KV_FP8 ? (SPARSE ? 0 : 64) : SPARSE ? 64 : 192;
  constexpr int RPW = MLA_KT / W;      // rows a wave copies
  constexpr int CPW = RPW + RPW / 8;   // copies: a row's latent values, 8 rows' rope
  constexpr int BUF = MLA_KT * (MLA_ROW + MLA_PE);
  __shared__ __attribute__((aligned(1024))) uint8_t S[2 * BUF];
  // scores on their way between the two waves of a pair
  __shared__ __attribute__((aligned(16))) f32x4v X[W][MLA_KT / 32][64];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15;
  const int l4 = lane >> 4;
  const int BS = 1 << bs_shift;

  // ---- this workgroup's run of tiles --------------------------------------------
  Run run = {(int)blockIdx.x, 0, 0, 1};
  if (tmp_acc == nullptr) {
    run.todo = (domain_of<SPARSE>(seq_lens, topk, max_topk, run.seq) + MLA_KT - 1) /
               MLA_KT;
    if (run.todo == 0) {  // no tokens: zeros, of this workgroup's heads
      const int h0 = blockIdx.y * (W * 8), n = min(W * 8, H - h0);
      for (int e = tid; e < n * (MLA_R / 4); e += W * 64)
        *reinterpret_cast<uint2*>(out + ((size_t)run.seq * H + h0) * MLA_R + e * 4) =
            make_uint2(0, 0);
    }
  } else {
    auto tiles_of = [&](int b) INL {
      return b < B ? (domain_of<SPARSE>(seq_lens, topk, max_topk, b) + MLA_KT - 1) / MLA_KT
                   : 0;
    };
    run = find_run<MLA_KT, MORE>(B, blockIdx.x, gridDim.x, tiles_of);
  }
  int seq = __builtin_amdgcn_readfirstlane(run.seq);
  int at = __builtin_amdgcn_readfirstlane(run.at);    // tile of the sequence
  int todo = __builtin_amdgcn_readfirstlane(run.todo);
  int done = 0;  // tiles of the run so far
  const int per = __builtin_amdgcn_readfirstlane(run.per);

  // two waves share 16 heads: each computes S^T of half of the tokens, and O^T of
  // half of the latent values
  const int head0 = (blockIdx.y * (W / 2) + (wid >> 1)) * 16;
  const int head = head0 + l15;
  const int d0 = (wid & 1) * (MLA_R / 2);

  // what a lane reads of a tile, in bytes: rows of S^T's operand (chunks l4 and
  // those at multiples of 4 from it) and of O^T's (chunks at multiples of 2)
  const int tr_row = 4 * l4 + (l15 >> 2);
  const uint32_t s_at = (uint32_t)(uintptr_t)(
      __attribute__((address_space(3))) const void*)S;
  const int qk_at = (wid & 1) * 32 * MLA_ROW + l15 * MLA_ROW +
                    (l4 ^ row_xor(l15)) * 16;
  const int pe_at = MLA_KT * MLA_ROW + (wid & 1) * 32 * MLA_PE + l15 * MLA_PE +
                    (l4 ^ rope_xor(l15)) * 16;
  const int tr_at = tr_row * MLA_ROW + d0 * 2 +
                    (((l15 & 3) >> 1) ^ row_xor(tr_row)) * 16 + (l15 & 1) * 8;
  // what a lane copies, in values: of row 8 g + i of the wave's (g the row's bit 3)
  // chunk (lane ^ row_xor), of the rope of 8 rows one chunk of row lane / 8
  const int bit3 = RPW == 8 ? wid & 1 : 0;

  bool first = true;
  while (todo > 0) {
    const int* btab = block_tables + (size_t)seq * max_blocks;
    const int L = seq_lens[seq];
    const int dom = domain_of<SPARSE>(seq_lens, topk, max_topk, seq);
    const bool listed = SPARSE && dom == max_topk &&
                        topk[(size_t)seq * max_topk] >= 0;
    const int* list = SPARSE ? topk + (size_t)seq * max_topk : nullptr;
    const int tiles = (dom + MLA_KT - 1) / MLA_KT;
    if (at >= tiles) {  // a sequence without tokens
      ++seq;
      at = 0;
      continue;
    }
    const int t0 = at;
    const int t1 = min(tiles, at + todo);
    if (tmp_acc != nullptr && t0 == 0 && tid == 0 && blockIdx.y == 0)
      part_runs(tmp_ml, gridDim.x, B, H)[seq] =
          make_int2(blockIdx.x, blockIdx.x + (done + tiles - 1) / per);

    bf16x8v qf[MLA_DK / 32];  // B operands: head l15, values 32 ks + 8 l4 + (0..7)
    f32x4v acc[MLA_DT] = {};
    float m = kHidden, l = 0.f;
    const float c = scale * kLog2e;

    // ---- copies --------------------------------------------------------------------
    // a list entry outside [0, L) stands for no token; its row reads token 0
    auto entry = [&](int j) INL { return j < dom ? list[j] : -1; };
    auto slot_of = [&](int tok) INL -> int {
      return (btab[tok >> bs_shift] << bs_shift) + (tok & (BS - 1));
    };
    // cache row (token slot) of tile row `lane`, listed; a sequence without tokens
    // has no page to look up
    auto listed_slot = [&](int t) INL {
      const int e = entry(t * MLA_KT + lane);
      return L > 0 ? slot_of(e >= 0 && e < L ? e : 0) : 0;
    };
    constexpr int ESZ = KV_FP8 ? 1 : 2;
    // Where tile t's rows of this wave lie: of every 8 the first one's slot (8 rows
    // lie in one page; rows past the end read a page that is there), or listed each
    // lane's row.
    int slots[RPW / 8], mine = 0;
    auto look_up = [&](int t) INL {
      if (listed) {
        mine = listed_slot(t);
        return;
      }
#pragma unroll
      for (int g = 0; g < RPW / 8; ++g)
        slots[g] = slot_of(min(t * MLA_KT + wid * RPW + g * 8, (L - 1) & ~7));
    };
    // copy i: use(i, place in the buffer, uniform base, values from there of a lane)
    auto copy_of = [&](int i, auto&& use) INL {
      const int g = i / 9, k = i % 9;      // k 0 .. 7: a row, 8: the rope of eight
      const int r0 = wid * RPW + g * 8;
      const int b3 = RPW == 8 ? bit3 : g;
      if (k < 8) {
        const int slot = SPARSE && listed
                             ? __builtin_amdgcn_readlane(mine, r0 + k)
                             : slots[g] + k;
        use(i, (r0 + k) * MLA_ROW,
            (const uint8_t*)cache + (int64_t)slot * (MLA_DK * ESZ),
            (lane ^ (2 * k) ^ b3 * 9) * 8);
      } else {
        const int r = lane >> 3;
        const int ch = (lane & 7) ^ (r & 6) ^ b3 * 5;
        if (SPARSE && listed) {
          const int slot = __shfl(mine, r0 + r, WAVE_SIZE);
          use(i, MLA_KT * MLA_ROW + r0 * MLA_PE,
              (const uint8_t*)cache + (int64_t)slot * (MLA_DK * ESZ),
              MLA_R + ch * 8);
        } else {
          use(i, MLA_KT * MLA_ROW + r0 * MLA_PE,
              (const uint8_t*)cache + (int64_t)slots[g] * (MLA_DK * ESZ),
              r * MLA_DK + MLA_R + ch * 8);
        }
      }
    };
    auto issue = [&](int i, int buf) INL {
      copy_of(i, [&](int i, int place, const uint8_t* base, int off) INL {
        const uint32_t at = s_at + buf * BUF + place;
        if (SPARSE && listed && i % 9 == 8) copy16(base + off * ESZ, at);
        else copy16(base, off * ESZ, at);
      });
    };
    uint64_t raw[KV_FP8 ? CPW : 1];
    auto fetch8 = [&] INL {
#pragma unroll
      for (int i = 0; i < (KV_FP8 ? CPW : 1); ++i)
        copy_of(i, [&](int i, int, const uint8_t* base, int off) INL {
          raw[KV_FP8 ? i : 0] = *(const uint64_t*)(base + (uint32_t)off);
        });
    };
    auto widen8 = [&](int buf) INL {
#pragma unroll
      for (int i = 0; i < (KV_FP8 ? CPW : 1); ++i)
        copy_of(i, [&](int i, int place, const uint8_t*, int) INL {
          int4 v;
          fp8x8_to_bf16x8(raw[KV_FP8 ? i : 0], 1.f,
                          reinterpret_cast<uint16_t*>(&v));
          *reinterpret_cast<int4*>(S + buf * BUF + place + lane * 16) = v;
        });
    };

    // ---- one tile --------------------------------------------------------------------
    // copy(n): the copies of the next tile that go with batch n of S^T's products
    auto compute = [&](int t, const int buf, auto&& copy) INL {
      uint8_t* T = S + buf * BUF;
      // rows that stand for a token, one bit each
      uint64_t alive = ~0ull;
      if (listed) {
        const int e = entry(t * MLA_KT + lane);
        alive = __ballot(e >= 0 && e < L);
      } else if (dom - t * MLA_KT < MLA_KT) {
        alive = (1ull << (dom - t * MLA_KT)) - 1;
      }
      if (alive != ~0ull) {  // the others may hold anything: weight 0 times it
        constexpr int CH = (MLA_ROW + MLA_PE) / 16;
        for (int i = tid; i < MLA_KT * CH; i += W * 64) {
          const int row = i / CH, ch = i % CH;
          if (!((alive >> row) & 1))
            *reinterpret_cast<int4*>(
                T + (ch < 64 ? row * MLA_ROW + ch * 16
                             : MLA_KT * MLA_ROW + row * MLA_PE + (ch - 64) * 16)) =
                make_int4(0, 0, 0, 0);
        }
        __syncthreads();
      }
      // Operands come in batches, the next one under way while this one's
      // products run: one read at a time would wait out the LDS each time.
      auto landed = [] INL {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        __builtin_amdgcn_sched_barrier(0);
      };
      constexpr int KB = KV_FP8 ? 1 : 3;  // of the 18 steps of S^T
      constexpr int NB = MLA_DK / 32 / KB;
      constexpr int TU = MLA_KT / 16;
      const bool on = head0 < H;  // a wave without heads copies only
      f32x4v s[TU] = {};
      if (on) {
        bf16x8v a[2][KB][TU / 2];
        auto fetch = [&](int n) INL {
#pragma unroll
          for (int i = 0; i < KB; ++i)
#pragma unroll
            for (int u = 0; u < TU / 2; ++u) {
              const int ks = n * KB + i;
              a[n & 1][i][u] = *reinterpret_cast<const bf16x8v*>(
                  T + (ks < 16 ? (qk_at ^ (ks & 3) * 64) + (ks >> 2) * 256 +
                                     u * 16 * MLA_ROW
                               : (pe_at ^ (ks & 1) * 64) + u * 16 * MLA_PE));
            }
        };
        fetch(0);
#pragma unroll
        for (int n = 0; n < NB; ++n) {
          landed();
          if (n + 1 < NB) fetch(n + 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < KB; ++i) {
#pragma unroll
            for (int u = 0; u < TU / 2; ++u)
              s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  a[n & 1][i][u], qf[n * KB + i], s[u], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            copy(n * KB + i);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
#pragma unroll
        for (int u = 0; u < TU / 2; ++u) X[wid][u][lane] = s[u];
      } else {
#pragma unroll
        for (int i = 0; i < NB * KB; ++i) copy(i);
      }
      // the scores of every wave are there; copies stay in flight
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (!on) return;
#pragma unroll
      for (int u = 0; u < TU; ++u)
        s[u] = X[(wid & ~1) + u / (TU / 2)][u % (TU / 2)][lane];
      // O^T's first operands are on their way beside the softmax
      constexpr int DB = 2;  // of a wave's latent tiles
      bf16x8v va[2][DB][TU / 2];
      auto fetch_v = [&](int n) INL {
#pragma unroll
        for (int i = 0; i < DB; ++i)
#pragma unroll
          for (int u = 0; u < TU / 2; ++u) {
            const int d = n * DB + i;
            uint8_t* src = T + (tr_at ^ (d & 7) * 32) + (d >> 3) * 256 +
                           u * 32 * MLA_ROW;
            const s16x4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) s16x4v*)src);
            const s16x4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) s16x4v*)(src + 16 * MLA_ROW));
            va[n & 1][i][u] =
                __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          }
      };
      float mx = kHidden;
      if (alive == ~0ull) {
#pragma unroll
        for (int u = 0; u < TU; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            s[u][r] *= c;
            mx = fmaxf(mx, s[u][r]);
          }
      } else {
        const uint64_t mine = alive >> (l4 * 4);
#pragma unroll
        for (int u = 0; u < TU; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            s[u][r] = (mine >> (u * 16 + r)) & 1 ? s[u][r] * c : kHidden;
            mx = fmaxf(mx, s[u][r]);
          }
      }
      mx = over_head(mx, [](float x, float y) { return fmaxf(x, y); });
      // rescaled when a maximum moved: its own weight is then 1, without rounding
      // (only when it moved by 2^8: 5 to 10% more error)
      if (__any(mx > m)) {
        const float m2 = fmaxf(m, mx);
        const float f = __builtin_amdgcn_exp2f(m - m2);
        m = m2;
        l *= f;
#pragma unroll
        for (int d = 0; d < MLA_DT; ++d) acc[d] *= f;
      }
      bf16x8v b[TU / 2];
#pragma unroll
      for (int n = 0; n < TU / 2; ++n) {
        float p[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          p[j] = __builtin_amdgcn_exp2f(s[2 * n + (j >> 2)][j & 3] - m);
          l += p[j];
        }
        uint32_t pk[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) pk[j] = pack_bf16(p[2 * j], p[2 * j + 1]);
        b[n] = *reinterpret_cast<const bf16x8v*>(pk);
      }

      // O^T: rows = 16 latent values, contraction over tokens 4 l4 + (0..3) and
      // 16 more: what lane group l4 of S^T holds
      fetch_v(0);
#pragma unroll
      for (int n = 0; n < MLA_DT / DB; ++n) {
        landed();
        if (n + 1 < MLA_DT / DB) fetch_v(n + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < TU / 2; ++u)
#pragma unroll
          for (int i = 0; i < DB; ++i)
            acc[n * DB + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                va[n & 1][i][u], b[u], acc[n * DB + i], 0, 0, 0);
      }
    };

    // ---- the run -----------------------------------------------------------------------
    // Behind a turn's first barrier this tile is in LDS, and every wave has left the
    // buffer that the next one goes to. Past the run's end nothing is copied.
    if (!first) __syncthreads();  // the buffers may still be read for the last sequence
    first = false;
    auto turn = [&](int t, const int buf) INL {
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this thread's copies
      __syncthreads();
      const bool more = t + 1 < t1;
      if (more) {
        look_up(t + 1);
        if constexpr (KV_FP8) fetch8();
      }
      compute(t, buf, [&](int n) INL {
        if constexpr (!KV_FP8) {
          constexpr int N = MLA_DK / 32;
          if (more)
#pragma unroll
            for (int i = 0; i < CPW; ++i)
              if (i * N / CPW == n) issue(i, buf ^ 1);
        }
      });
      if constexpr (KV_FP8)
        if (more) widen8(buf ^ 1);
    };
    look_up(t0);
    if constexpr (KV_FP8) {
      fetch8();
      widen8(0);
    } else {
#pragma unroll
      for (int i = 0; i < CPW; ++i) issue(i, 0);
    }
    // behind the first tile's copies, whose way is the longer one
    {
      const size_t row = (size_t)seq * H + min(head, H - 1);
#pragma unroll
      for (int ks = 0; ks < MLA_DK / 32; ++ks) {
        const int k = ks * 32 + l4 * 8;
        qf[ks] = ks < MLA_R / 32
                     ? *(const bf16x8v*)(q_latent + row * MLA_R + k)
                     : *(const bf16x8v*)(q_pe + row * MLA_DR + k - MLA_R);
      }
    }
    for (int t = t0; t < t1;) {
      turn(t, 0);
      if (++t >= t1) break;
      turn(t, 1);
      ++t;
    }

    // ---- results: column = head, rows = latent values --------------------------------
    l = over_head(l, [](float x, float y) { return x + y; });
    if (head < H) {
      if (t0 == 0 && t1 == tiles) {
        const float inv = 1.f / l;
        uint16_t* o = out + ((size_t)seq * H + head) * MLA_R + d0 + l4 * 4;
#pragma unroll
        for (int d = 0; d < MLA_DT; ++d) {
          uint2 v;
          v.x = pack_bf16(acc[d][0] * inv, acc[d][1] * inv);
          v.y = pack_bf16(acc[d][2] * inv, acc[d][3] * inv);
          *reinterpret_cast<uint2*>(o + d * 16) = v;
        }
      } else {
        // a run has one part of a sequence, and one of each more sequence that it meets:
        // runs and sequences both advance, so their sum names a part
        const size_t part = ((size_t)blockIdx.x + seq) * H + head;
        float* o = tmp_acc + part * MLA_R + d0 + l4 * 4;
#pragma unroll
        for (int d = 0; d < MLA_DT; ++d)
          *reinterpret_cast<f32x4v*>(o + d * 16) = acc[d];
        if (l4 == 0 && d0 == 0) {
          tmp_ml[part * 2] = m;  // in units of log2
          tmp_ml[part * 2 + 1] = l;
        }
      }
    }
    todo -= t1 - t0;
    done += t1 - t0;
    ++seq;
    at = 0;
  }
}

// ---- an fp8 cache, more than 32 heads ---------------------------------------------
// Four waves, 64 heads: 32 a pair of waves, on 32x32 matrix instructions, so that an
// operand row read from LDS serves 32 heads instead of 16. A wave computes S^T over
// half of the 576 values, for which it holds the heads' Q, adds the other wave's half,
// and takes half of the latent values of O^T: 200 registers of state, so one wave a
// SIMD. Tiles of 32 tokens in a ring of four, three of them on their way. In turn t
// the products of S^T of tile t + 1 stand beside tile t's softmax.
// us of a call, mla_decode_kernel of eight waves (16 heads a pair, tiles of 64) / so: 64
// heads, 4 x 21,111 tokens 42.7 / 41.4, 2 x 100,000 66.1 / 63.9; 128 heads, 20 x 9,000 100.5 /
// 97.3, 70 x 3,000 121 / 118. With a bf16 cache the eight waves are as fast or faster: 64
// heads, 20 x 9,000 54.4 / 56.1, 2 x 18,786 30.9 / 31.8; 128 heads, 16 x 16,384 119 / 122, 40
// x 4,000 77 / 80.
__global__ __launch_bounds__(256, 1) void mla_decode_wide_kernel(
    uint16_t* __restrict__ out,             // [B, H, R]
    float* __restrict__ tmp_acc,            // [parts, H, R]; null: a workgroup
    float* __restrict__ tmp_ml,             // [parts, H, 2]      a sequence
    const uint16_t* __restrict__ q_latent,  // [B, H, R]
    const uint16_t* __restrict__ q_pe,      // [B, H, DR]
    const void* __restrict__ cache,         // [NB, BS, R+DR] fp8(e4m3)
    const int* __restrict__ block_tables,   // [B, max_blocks]
    const int* __restrict__ seq_lens, const int B, const int max_blocks,
    const int H, const int bs_shift, const float scale) {
  constexpr int MORE = 288;  // see find_run
  constexpr int BUF = MLA_WT * (MLA_ROW + MLA_PE);
  constexpr int PE = MLA_WT * MLA_ROW;  // of a buffer's rotated values
  constexpr int RING = 4;
  constexpr int CPW = 9;                // copies a wave: 8 rows, their rotated values
  constexpr int QS = 18;                // steps of 16 values of S^T a wave
  constexpr int DT = 8;                 // tiles of 32 latent values of O^T a wave
  __shared__ __attribute__((aligned(1024))) uint8_t S[RING * BUF];
  // sums over half of the values on their way to the other wave of a pair
  __shared__ __attribute__((aligned(16))) f32x4v X[4][4][64];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l31 = lane & 31, half = lane >> 5;
  const int BS = 1 << bs_shift;

  Run run = {(int)blockIdx.x, 0, 0, 1};
  if (tmp_acc == nullptr) {
    run.todo = (max(seq_lens[run.seq], 0) + MLA_WT - 1) / MLA_WT;
    if (run.todo == 0) {  // no tokens: zeros, of this workgroup's heads
      const int h0 = blockIdx.y * 64, n = min(64, H - h0);
      for (int e = tid; e < n * (MLA_R / 4); e += 256)
        *reinterpret_cast<uint2*>(out + ((size_t)run.seq * H + h0) * MLA_R + e * 4) =
            make_uint2(0, 0);
    }
  } else {
    auto tiles_of = [&](int b) INL {
      return b < B ? (max(seq_lens[b], 0) + MLA_WT - 1) / MLA_WT : 0;
    };
    run = find_run<MLA_WT, MORE>(B, blockIdx.x, gridDim.x, tiles_of);
  }
  int seq = __builtin_amdgcn_readfirstlane(run.seq);
  int at = __builtin_amdgcn_readfirstlane(run.at);    // tile of the sequence
  int todo = __builtin_amdgcn_readfirstlane(run.todo);
  int done = 0;  // tiles of the run so far
  const int per = __builtin_amdgcn_readfirstlane(run.per);

  const int h = wid & 1;  // which half of the values
  const int head = (blockIdx.y * 2 + (wid >> 1)) * 32 + l31;

  // Chunk c of row r of a tile lies at c ^ wide_xor(r), of its rotated values at c ^
  // ((r >> 1) & 7). 16-byte reads of one chunk go by rows {0-3, 12-15, 20-23, 24-27}
  // and the others, which differ in both; transposing reads take four neighbouring
  // chunks of four rows, which differ in bits 2 and 3 of wide_xor.
  auto wide_xor = [](int r) INL { return (r & 3) * 4 + (r >> 2 & 3); };
  const int qk_at = l31 * MLA_ROW + h * 512 + (half ^ wide_xor(l31)) * 16;
  const int pe_at = PE + l31 * MLA_PE + ((4 * h + half) ^ (l31 >> 1 & 7)) * 16;
  const int tr_row = 4 * half + (l15 >> 2);
  const int tr_at = tr_row * MLA_ROW + h * 512 +
                    ((2 * (lane >> 4 & 1) + (l15 >> 1 & 1)) ^ wide_xor(tr_row)) * 16 +
                    (l15 & 1) * 8;
  // copy i of a wave: row 8 wid + i's latent values, or of its 8 rows the rotated ones
  uint32_t from[CPW];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    from[i] = i * MLA_DK + (lane ^ wide_xor(wid * 8 + i)) * 8;
  from[8] = (lane >> 3) * MLA_DK + MLA_R +
            ((lane & 7) ^ ((wid * 8 + (lane >> 3)) >> 1 & 7)) * 8;
  auto place = [&](int i) INL {
    return i < 8 ? (wid * 8 + i) * MLA_ROW : PE + wid * 8 * MLA_PE;
  };

  bool first = true;
  while (todo > 0) {
    // Q first: its many rows are on their way while length and pages are looked up
    bf16x8v qf[QS];  // head l31, values 16 i + 8 half of this wave's
    {
      const size_t row = (size_t)seq * H + min(head, H - 1);
#pragma unroll
      for (int i = 0; i < QS; ++i)
        qf[i] = i < 16
                    ? *(const bf16x8v*)(q_latent + row * MLA_R + h * 256 + i * 16 + half * 8)
                    : *(const bf16x8v*)(q_pe + row * MLA_DR + h * 32 + (i - 16) * 16 +
                                        half * 8);
    }
    const int L = seq_lens[seq];
    const int tiles = (max(L, 0) + MLA_WT - 1) / MLA_WT;
    if (at >= tiles) {  // a sequence without tokens
      ++seq;
      at = 0;
      continue;
    }
    const auto* btab = (const __attribute__((address_space(4))) int*)(
        block_tables + (size_t)seq * max_blocks);
    const int t0 = at;
    const int t1 = min(tiles, at + todo);
    if (tmp_acc != nullptr && t0 == 0 && tid == 0 && blockIdx.y == 0)
      part_runs(tmp_ml, gridDim.x, B, H)[seq] =
          make_int2(blockIdx.x, blockIdx.x + (done + tiles - 1) / per);

    // ---- copies: tile t goes to place t - t0 of the ring -------------------------------
    // 8 rows lie in one page; rows past the end read a page that is there
    auto token_of = [&](int t) INL { return min(t * MLA_WT + wid * 8, (L - 1) & ~7); };
    auto page_of = [&](int t) INL { return btab[token_of(t) >> bs_shift]; };
    auto base_of = [&](int t, int page) INL {
      const int slot = (page << bs_shift) + (token_of(t) & (BS - 1));
      return (const uint8_t*)cache + (int64_t)slot * MLA_DK;
    };
    uint64_t raw[2][CPW];  // two tiles on their way
    auto fetch8 = [&](uint64_t (&r)[CPW], int t, int page) INL {
      const uint8_t* base = base_of(t, page);
#pragma unroll
      for (int i = 0; i < CPW; ++i)
        r[i] = *(const uint64_t*)(base + from[i]);
    };
    auto widen8 = [&](const uint64_t (&r)[CPW], int t) INL {
      uint8_t* T = S + ((t - t0) & (RING - 1)) * BUF + lane * 16;
#pragma unroll
      for (int i = 0; i < CPW; ++i) {
        bf16x8n v;  // every e4m3 number is one of bf16
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const auto two = j & 1
              ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((uint32_t)(r[i] >> 32 * (j >> 1)),
                                                          1.f, true)
              : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((uint32_t)(r[i] >> 32 * (j >> 1)),
                                                          1.f, false);
          v[2 * j] = two[0];
          v[2 * j + 1] = two[1];
        }
        *reinterpret_cast<bf16x8n*>(T + place(i)) = v;
      }
    };

    f32x16v acc[DT] = {};
    f32x16v sc[2];  // scores of a tile and of the next one
    float m = kHidden, l = 0.f;
    const float c = fmaxf(fabsf(scale) * kLog2e, 1e-30f);  // the sign: Q's
    bf16x8v b[2];   // the weights, operands of O^T
    float f = 1.f;  // of O^T so far

    auto meet = [] INL {  // copies stay in flight
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
    // rows of the last tile that stand for no token may hold anything: weight 0 times it
    auto clear_rest = [&](int t) INL {
      const int n = L - t * MLA_WT;
      if (n >= MLA_WT || n <= 0) return;
      constexpr int CH = (MLA_ROW + MLA_PE) / 16;
      uint8_t* T = S + ((t - t0) & (RING - 1)) * BUF;
      for (int i = n * CH + tid; i < MLA_WT * CH; i += 256) {
        const int row = i / CH, ch = i % CH;
        *reinterpret_cast<int4*>(
            T + (ch < 64 ? row * MLA_ROW + ch * 16
                         : PE + row * MLA_PE + (ch - 64) * 16)) = make_int4(0, 0, 0, 0);
      }
      __syncthreads();
    };

    // S^T over this wave's values; between(i): what goes with product i. One wave a
    // SIMD: operands are asked for two batches ahead.
    auto scores = [&](int t, f32x16v& r, auto&& between) INL {
      const uint8_t* T = S + ((t - t0) & (RING - 1)) * BUF;
      constexpr int KB = 3;
      bf16x8v a[3][KB];
      auto fetch = [&](int n) INL {
#pragma unroll
        for (int i = 0; i < KB; ++i) {
          const int ks = n * KB + i;
          a[n % 3][i] = *reinterpret_cast<const bf16x8v*>(
              T + (ks < 16 ? (qk_at ^ (ks & 7) * 32) + (ks >> 3) * 256
                           : pe_at ^ (ks & 1) * 32));
        }
      };
      r = f32x16v{};
      fetch(0);
      fetch(1);
#pragma unroll
      for (int n = 0; n < QS / KB; ++n) {
        __builtin_amdgcn_sched_barrier(0);
        if (n + 2 < QS / KB) fetch(n + 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < KB; ++i) {
          r = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[n % 3][i], qf[n * KB + i], r, 0, 0,
                                                      0);
          __builtin_amdgcn_sched_barrier(0);
          between(n * KB + i);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    auto publish = [&](const f32x16v& r) INL {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        X[wid][q][lane] = f32x4v{r[4 * q], r[4 * q + 1], r[4 * q + 2], r[4 * q + 3]};
    };

    // ---- the softmax of a tile, in 18 pieces ---------------------------------------------
    // token 8 q + 4 half + r of the tile in s[4 q + r]
    float mx;
    auto soften = [&](int i, f32x16v& s, const f32x4v (&x)[4]) INL {
      if (i < 4) {
#pragma unroll
        for (int r = 0; r < 4; ++r) s[4 * i + r] += x[i][r];
        const float a = fmaxf(fmaxf(s[4 * i], s[4 * i + 1]), s[4 * i + 2]);
        mx = i == 0 ? fmaxf(a, s[3]) : fmaxf(fmaxf(mx, a), s[4 * i + 3]);
      } else if (i == 4) {
        const auto o = __builtin_amdgcn_permlane32_swap(
            __float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = fmaxf(__uint_as_float(o[0]), __uint_as_float(o[1])) * c;
        // a new maximum's own weight is 1, without rounding (m moved only by 2^8 and
        // more: 2 to 13% more error)
        const float m2 = fmaxf(m, mx);
        f = __builtin_amdgcn_exp2f(m - m2);
        m = m2;
        l *= f;
      } else if (i < 13) {
        const int e = (i - 5) * 2;
        const float p0 = __builtin_amdgcn_exp2f(fmaf(s[e], c, -m));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(s[e + 1], c, -m));
        l += p0;  // in fp32: only the products' operands are rounded
        l += p1;
        const uint32_t pk = pack_bf16(p0, p1);
        auto w = __builtin_bit_cast(u32x4v, b[e >> 3]);
        w[e >> 1 & 3] = pk;
        b[e >> 3] = __builtin_bit_cast(bf16x8v, w);
      }
    };

    // O^T: rows = 32 latent values, contraction over tokens 16 u + 4 half + (0..3) and
    // 8 more: what this half of S^T's lanes holds
    bf16x8v va[3][2];
    auto fetch_v = [&](int t, int d) INL {
      uint8_t* T = S + ((t - t0) & (RING - 1)) * BUF;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        uint8_t* src = T + (d >> 2) * 256 + u * 16 * MLA_ROW;
        const s16x4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4v*)(src + (tr_at ^ (d & 3) * 64)));
        const s16x4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4v*)(
                src + 8 * MLA_ROW + (tr_at ^ ((d & 3) * 64 + 32))));
        va[d % 3][u] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
    };
    auto weigh = [&](int t) INL {  // behind fetch_v of 0 and 1
      acc[0] *= f;
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        __builtin_amdgcn_sched_barrier(0);
        if (d + 2 < DT) fetch_v(t, d + 2);
        __builtin_amdgcn_sched_barrier(0);
        acc[d] =
            __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[d % 3][0], b[0], acc[d], 0, 0, 0);
        if (d + 1 < DT) acc[d + 1] *= f;
        acc[d] =
            __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[d % 3][1], b[1], acc[d], 0, 0, 0);
      }
    };

    // ---- the run -----------------------------------------------------------------------
    if (scale < 0.f)
#pragma unroll
      for (int i = 0; i < QS; ++i) qf[i] ^= (short)0x8000;
    // Q is read by products alone: in the registers that only those take as operands. It
    // is there before the copies are asked for, as a wait for it would be one for them
#pragma unroll
    for (int i = 0; i < QS; ++i) asm volatile("" : "+a"(qf[i]));
    if (!first) __syncthreads();  // the buffers may still be read for the last sequence
    first = false;
    fetch8(raw[0], t0, page_of(t0));
    fetch8(raw[1], min(t0 + 1, t1 - 1), page_of(min(t0 + 1, t1 - 1)));
    // the first tile's scores
    widen8(raw[0], t0);
    const int t2 = min(t0 + 2, t1 - 1);
    fetch8(raw[0], t2, page_of(t2));
    widen8(raw[1], t0 + 1);
    meet();
    clear_rest(t0);
    scores(t0, sc[0], [](int) {});
    publish(sc[0]);

    // Turn t. Behind its first barrier tile t + 1 is in LDS, both halves of S^T of tile
    // t are there, and every wave has left the place that tile t + 2 goes to. Past the
    // run's end copies and products go on with its last tile: one loop for all turns, as
    // instructions that are not in the cache yet cost a run of few tiles 1 us and more.
    int page = page_of(min(t0 + 3, t1 - 1));  // of the tile that the next turn copies
    auto turn = [&](int t, auto even) INL {
      constexpr int P = decltype(even)::value;
      meet();
      f32x4v x[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) x[q] = X[wid ^ 1][q][lane];
      const int rest = L - t * MLA_WT;
      if (rest < MLA_WT)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            x[q][r] = 8 * q + 4 * half + r < rest ? x[q][r] : -3e38f;
      fetch8(raw[P ^ 1], min(t + 3, t1 - 1), page);
      clear_rest(t + 1);
      scores(t + 1, sc[P ^ 1], [&](int i) INL {
        soften(i, sc[P], x);
        // on their way to behind the barrier
        if (i == 15) fetch_v(t, 0);
        if (i == 16) fetch_v(t, 1);
        if (i == 17) page = page_of(min(t + 4, t1 - 1));
      });
      meet();  // every wave has the other's half of tile t
      publish(sc[P ^ 1]);
      weigh(t);
      widen8(raw[P], t + 2);
    };
    for (int t = t0;;) {
      turn(t, Int<0>{});
      if (++t >= t1) break;
      turn(t, Int<1>{});
      if (++t >= t1) break;
    }

    // ---- results: column = head, rows = latent values --------------------------------
    {
      const auto o = __builtin_amdgcn_permlane32_swap(
          __float_as_uint(l), __float_as_uint(l), false, false);
      l = __uint_as_float(o[0]) + __uint_as_float(o[1]);
    }
    if (head < H) {
      const int d0 = h * 256 + half * 4;
      if (t0 == 0 && t1 == tiles) {
        const float inv = 1.f / l;
        uint16_t* o = out + ((size_t)seq * H + head) * MLA_R + d0;
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            uint2 v;
            v.x = pack_bf16(acc[d][4 * q] * inv, acc[d][4 * q + 1] * inv);
            v.y = pack_bf16(acc[d][4 * q + 2] * inv, acc[d][4 * q + 3] * inv);
            *reinterpret_cast<uint2*>(o + d * 32 + q * 8) = v;
          }
      } else {
        // a run has one part of a sequence, and one of each more sequence that it meets:
        // runs and sequences both advance, so their sum names a part
        const size_t part = ((size_t)blockIdx.x + seq) * H + head;
        float* o = tmp_acc + part * MLA_R + d0;
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4v*>(o + d * 32 + q * 8) =
                f32x4v{acc[d][4 * q], acc[d][4 * q + 1], acc[d][4 * q + 2],
                       acc[d][4 * q + 3]};
        if (half == 0 && h == 0) {
          tmp_ml[part * 2] = m;  // in units of log2
          tmp_ml[part * 2 + 1] = l;
        }
      }
    }
    todo -= t1 - t0;
    done += t1 - t0;
    ++seq;
    at = 0;
  }
}

// Adds up the parts of the sequences that several runs share: four groups of 128
// threads, a thread four values. Few sequences (BY_HEAD false) have many parts:
// a workgroup a head, the groups share its parts. Many have few: a group a head.
// Measured, 64 heads x 4 sequences x 64 parts: 8.5 us (54 us as a serial loop
// over the parts); 128 heads x 256 sequences of two parts: 28 us.
template <bool SPARSE, bool BY_HEAD>
__global__ __launch_bounds__(512) void mla_reduce_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ tmp_acc,
    const float* __restrict__ tmp_ml, const int* __restrict__ seq_lens,
    const int* __restrict__ topk, const int max_topk, const int B, const int H,
    const int runs) {
  const int seq = blockIdx.y;
  const int tid = threadIdx.x;
  const int lane = tid & 63, grp = tid >> 7;
  const int head = BY_HEAD ? blockIdx.x * 4 + grp : blockIdx.x;
  const int2 range = part_runs(const_cast<float*>(tmp_ml), runs, B, H)[seq];
  if (domain_of<SPARSE>(seq_lens, topk, max_topk, seq) == 0) {  // no tokens: zeros
    if (head < H)
      for (int d = (BY_HEAD ? tid & 127 : tid) * 4; d < MLA_R;
           d += (BY_HEAD ? 128 : 512) * 4)
        *reinterpret_cast<uint2*>(out + ((size_t)seq * H + head) * MLA_R + d) =
            make_uint2(0, 0);
    return;
  }
  const int r0 = range.x, r1 = range.y;
  if (r0 == r1) return;  // finished by its run

  __shared__ f32x4v sums[4][128];
  __shared__ float wt[BY_HEAD ? 4 : 1][MLA_MAX_RUNS];
  const int parts = r1 - r0 + 1;
  const bool on = head < H;
  const size_t first_part = ((size_t)r0 + seq) * H + (on ? head : 0);
  // a thread's first parts, on their way beside the weights
  constexpr int STEP = BY_HEAD ? 1 : 4, AHEAD = 8;
  const int d = (tid & 127) * 4, mine = BY_HEAD ? 0 : grp;
  const float* src = tmp_acc + first_part * MLA_R + d;
  f32x4v v[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
    v[i] = *reinterpret_cast<const f32x4v*>(
        src + (size_t)min(mine + i * STEP, parts - 1) * H * MLA_R);
  // the weights, worked out by each wave for itself, written by one of them
  float M = kHidden, l = 0.f;
  for (int r = lane; r < parts; r += 64)
    M = fmaxf(M, tmp_ml[(first_part + (size_t)r * H) * 2]);
  M = wave_reduce_max(M);
  for (int r = lane; r < parts; r += 64) {
    const float* ml = tmp_ml + (first_part + (size_t)r * H) * 2;
    const float w = __builtin_amdgcn_exp2f(ml[0] - M);
    l += ml[1] * w;
    if ((BY_HEAD ? tid & 127 : tid) < 64) wt[BY_HEAD ? grp : 0][r] = w;
  }
  l = wave_reduce_sum(l);
  __syncthreads();
  f32x4v s = {0.f, 0.f, 0.f, 0.f};
  auto add = [&](f32x4v part, int r) {
    const float w = wt[BY_HEAD ? grp : 0][r];
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = fmaf(part[i], w, s[i]);
  };
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
    if (mine + i * STEP < parts) add(v[i], mine + i * STEP);
#pragma unroll 8
  for (int r = mine + AHEAD * STEP; r < parts; r += STEP)
    add(*reinterpret_cast<const f32x4v*>(src + (size_t)r * H * MLA_R), r);
  if (!BY_HEAD) {
    sums[grp][tid & 127] = s;
    __syncthreads();
    if (grp > 0) return;
    s = sums[0][tid] + sums[1][tid] + sums[2][tid] + sums[3][tid];
  }
  if (!on) return;
  const float inv = 1.f / l;
  *reinterpret_cast<uint2*>(out + ((size_t)seq * H + head) * MLA_R + d) = make_uint2(
      pack_bf16(s[0] * inv, s[1] * inv), pack_bf16(s[2] * inv, s[3] * inv));
}

// Runs the tiles are dealt to; 0: every sequence has a workgroup of its own.
// One workgroup a CU: its tiles (144 KB) fill the LDS.
extern "C" int mla_decode_runs(int B, int H, int max_domain) {
  const int blocks = ceil_div(H, 64);
  if (max_domain <= 256) return 0;
  return MLA_MAX_RUNS / blocks > 1 ? MLA_MAX_RUNS / blocks : 1;
}

extern "C" void launch_mla_paged_attention_decode(
    void* out, const void* q_latent, const void* q_pe, const void* cache,
    const int* block_tables, const int* seq_lens, int B, int H, int R, int DR,
    int BS, int max_blocks, float scale, int runs, float* tmp_acc,
    float* tmp_ml, const int* topk_indices, int max_topk, bool kv_fp8,
    hipStream_t stream, bool* launched) {
  *launched = false;
  if (R != MLA_R || DR != MLA_DR) return;  // DeepSeek V2/V3/R1/K2 geometry
  if (BS != 16 && BS != 32 && BS != 64) return;
  const int shift = __builtin_ctz(BS);
  const int waves = H > 32 ? 8 : 4;
  dim3 grid(runs > 0 ? runs : B, ceil_div(H, waves * 8), 1);

#define MLA_ARGS                                                               \
  (uint16_t*)out, tmp_acc, tmp_ml, (const uint16_t*)q_latent,                  \
      (const uint16_t*)q_pe, cache, block_tables, seq_lens
  auto decode = [&](auto w, auto fp8, auto sparse) {
    mla_decode_kernel<decltype(w)::value, decltype(fp8)::value, decltype(sparse)::value>
        <<<grid, decltype(w)::value * 64, 0, stream>>>(
            MLA_ARGS, topk_indices, max_topk, B, max_blocks, H, shift, scale);
  };
  auto reduce = [&](auto sparse) {
    constexpr bool SP = decltype(sparse)::value;
    if (runs <= 0) return;
    if (runs >= 16 * B)
      mla_reduce_kernel<SP, false><<<dim3(H, B, 1), 512, 0, stream>>>(
          (uint16_t*)out, tmp_acc, tmp_ml, seq_lens, topk_indices, max_topk, B, H, runs);
    else
      mla_reduce_kernel<SP, true><<<dim3(ceil_div(H, 4), B, 1), 512, 0, stream>>>(
          (uint16_t*)out, tmp_acc, tmp_ml, seq_lens, topk_indices, max_topk, B, H, runs);
  };
  using True = std::true_type;
  using False = std::false_type;
  if (topk_indices != nullptr) {
    if (waves == 8 && kv_fp8) decode(Int<8>{}, True{}, True{});
    else if (waves == 8) decode(Int<8>{}, False{}, True{});
    else if (kv_fp8) decode(Int<4>{}, True{}, True{});
    else decode(Int<4>{}, False{}, True{});
    reduce(True{});
  } else if (H > 32) {
    if (kv_fp8)
      mla_decode_wide_kernel<<<grid, 256, 0, stream>>>(MLA_ARGS, B, max_blocks, H, shift,
                                                       scale);
    else
      decode(Int<8>{}, False{}, False{});
    reduce(False{});
  } else {
    if (kv_fp8) decode(Int<4>{}, True{}, False{});
    else decode(Int<4>{}, False{}, False{});
    reduce(False{});
  }
#undef MLA_ARGS
  *launched = true;
}
