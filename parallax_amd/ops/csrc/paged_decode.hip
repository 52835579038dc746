// Decode attention over the paged K/V cache for gfx950.
//
//   S^T[32 tok x 16 q] = K . Q^T    O^T[D x 16 q] += V^T . P
// A key/value head's query group (at most 16 heads) are the columns; V is stored
// transposed ([NB, Hk, D, BS]), so both operands are rows of the cache.
//
// Every wave is on its own: it goes through tiles of 32 tokens, whose K and V are
// copied global -> LDS directly, 1 KB of neighbouring memory a copy, into its own
// two places. A place is filled again as soon as its operands are in registers, so
// that 8 to 16 KB a wave are always on their way; no barrier but where the waves'
// sums are added, at the end of a sequence. K rows are taken in an order in which
// the accumulators of S^T are the operand of the second product, so P stays in
// registers. 16-byte chunks are XOR-swizzled to spread both reads over the banks.
// An fp8 cache is widened between LDS and the products (exactly: the scales are
// applied to the sums).
//
// Work is split by tokens, not by sequences: a unit is 32 tokens a wave, the units
// of all sequences form one list, of which every workgroup of a key/value head
// takes an equal run. Lengths are read on the device, so a captured step balances
// for any lengths. A sequence that lies in one run is finished there; of the
// others the runs leave fp32 parts that a second kernel adds up. Short contexts
// take a workgroup a sequence and head, of more waves where there are few.
//
// What bounds it: large batches the cache's stream, 128 x 8 heads x 128 of 1,024 to
// 4,096 tokens (1.39 GB) 253 us or 5.5 TB/s (before, barriers in every tile and
// fixed partitions: 272); 64-wide fp8 heads the instructions of a tile beside its few bytes, 200 x 8
// of 3,001 87 us (196); one sequence two round trips and the launches, 8 heads of
// 1,000 9.4 us (11.8), of 32,000 34 us (84).
//
// Reference analogue: parallax_extensions/kernels/paged_attention/ (Metal, v1/v2).

#include <type_traits>

#include "common.h"
#include "decode_common.h"

#define PD_KT 32           // tokens a tile
#define PD_MAX_RUNS 512

#define INL __attribute__((always_inline))

typedef unsigned int u32x2v __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4v __attribute__((ext_vector_type(4)));

namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kHidden = -__builtin_inff();  // score of a key that is not seen
constexpr float kLowest = -1e30f;              // where a maximum starts

DEVINL void copy16_to_lds(const void* src, void* dst) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)src,
      (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

template <int N>
DEVINL void wait_copies() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N & 48) << 10));
  asm volatile("" ::: "memory");
}

DEVINL uint32_t lds_at(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

// Operands out of LDS, each block with its own wait: before plain loads the
// compiler waits for every copy in flight.
#define RD "ds_read_b128 "
template <int OFF>
DEVINL void read2(u32x4v (&v)[2], uint32_t a) {
  asm volatile(RD "%0, %2\n\t" RD "%1, %2 offset:%3\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]) : "v"(a), "n"(OFF) : "memory");
}
template <int OFF>
DEVINL void read4(u32x4v (&v)[4], uint32_t a, uint32_t b) {
  asm volatile(RD "%0, %4\n\t" RD "%1, %4 offset:%6\n\t" RD "%2, %5\n\t"
               RD "%3, %5 offset:%6\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
               : "v"(a), "v"(b), "n"(OFF) : "memory");
}
template <int OFF>
DEVINL void read8(u32x4v (&v)[8], uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  asm volatile(RD "%0, %8\n\t" RD "%1, %8 offset:%12\n\t" RD "%2, %9\n\t"
               RD "%3, %9 offset:%12\n\t" RD "%4, %10\n\t"
               RD "%5, %10 offset:%12\n\t" RD "%6, %11\n\t"
               RD "%7, %11 offset:%12\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]),
                 "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
               : "v"(a), "v"(b), "v"(c), "v"(d), "n"(OFF) : "memory");
}
DEVINL void read_rows(u32x4v (&v)[4], uint32_t a) {
  asm volatile(RD "%0, %4\n\t" RD "%1, %4 offset:1024\n\t"
               RD "%2, %4 offset:2048\n\t" RD "%3, %4 offset:3072\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
               : "v"(a) : "memory");
}
DEVINL void read_rows(u32x4v (&v)[8], uint32_t a) {
  asm volatile(RD "%0, %8\n\t" RD "%1, %8 offset:1024\n\t"
               RD "%2, %8 offset:2048\n\t" RD "%3, %8 offset:3072\n\t"
               RD "%4, %8 offset:4096\n\t" RD "%5, %8 offset:5120\n\t"
               RD "%6, %8 offset:6144\n\t" RD "%7, %8 offset:7168\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]),
                 "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
               : "v"(a) : "memory");
}
#undef RD
#define RD "ds_read_b64 "
DEVINL void read_rows(u32x2v (&v)[4], uint32_t a) {
  asm volatile(RD "%0, %4\n\t" RD "%1, %4 offset:512\n\t"
               RD "%2, %4 offset:1024\n\t" RD "%3, %4 offset:1536\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
               : "v"(a) : "memory");
}
DEVINL void read_rows(u32x2v (&v)[8], uint32_t a) {
  asm volatile(RD "%0, %8\n\t" RD "%1, %8 offset:512\n\t"
               RD "%2, %8 offset:1024\n\t" RD "%3, %8 offset:1536\n\t"
               RD "%4, %8 offset:2048\n\t" RD "%5, %8 offset:2560\n\t"
               RD "%6, %8 offset:3072\n\t" RD "%7, %8 offset:3584\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]),
                 "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
               : "v"(a) : "memory");
}
#undef RD

// 8 e4m3 values to bf16, exact
DEVINL bf16x8v widen(uint32_t lo, uint32_t hi) {
  u32x4v r;
  r[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, false));
  r[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, true));
  r[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, false));
  r[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, true));
  return __builtin_bit_cast(bf16x8v, r);
}

// Where chunk c of a row lies: at c ^ swz(row), linear over xor in the row's bits.
// 16 lanes read at a time (0-3, 12-15 and 20-23, 24-27, ..): rows of two lane
// groups, which differ in bit 0 of the chunk. four(): 0, 2, 3, 1.
DEVINL constexpr int four(int a) { return ((a & 1) << 1) ^ ((a >> 1) & 1) * 3; }
template <int CPR>  // chunks a K row; its rows go 8 (l15 / 4) + (l15 & 3)
DEVINL constexpr int swz_k(int r) {
  return CPR == 16 ? ((r >> 3) & 3) * 4 + (r & 3)
         : CPR == 8 ? ((r >> 3) & 3) * 2 + ((r >> 1) & 1)
                    : four((r >> 3) & 3);
}
template <bool FP8>  // V rows: 4 chunks (bf16), 2 (fp8)
DEVINL constexpr int swz_v(int d) {
  return FP8 ? (d >> 3) & 1 : four((d >> 2) & 3);
}

// units of u tokens of a sequence of n: those from its window's first token on
DEVINL int units_of(int n, int window, int u) {
  const int lo = window > 0 ? max(0, n - window) : 0;
  return n > 0 ? (n + u - 1) / u - lo / u : 0;
}

// inclusive sum over the lanes of a wave
DEVINL int scan64(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(v, o, WAVE_SIZE);
    if (lane >= o) v += t;
  }
  return v;
}

DEVINL int run_length(int total, int runs) {
  return max((total + runs - 1) / runs, 1);
}

// the first and the last run of each sequence, behind the parts' maxima and sums
DEVINL int2* part_runs(float* tmp_ml, int runs, int B, int Hq) {
  return reinterpret_cast<int2*>(tmp_ml + ((size_t)runs + B) * Hq * 2);
}

// Run `run` of the list of all sequences' units: its length, the sequence that
// holds its first unit, that unit's place there, and the length of a full run. Found by
// one wave: lanes sum equal groups of sequences, the group's sequences are then looked at.
DEVINL int find_run(const int* seq_lens, int window, int u, int B, int run,
                    int runs, int* seq, int* at, int* per_run) {
  const int lane = threadIdx.x & 63;
  const int per_lane = (B + 63) / 64;
  int n = 0;
  for (int i = 0; i < per_lane; ++i) {
    const int b = lane * per_lane + i;
    n += b < B ? units_of(seq_lens[b], window, u) : 0;
  }
  const int sum = scan64(n);
  const int total = __shfl(sum, 63, WAVE_SIZE);
  const int per = run_length(total, runs);
  *per_run = per;
  const int begin = run * per;
  *seq = 0;
  *at = 0;
  if (begin >= total) return 0;
  const int src = __ffsll(__ballot(sum > begin)) - 1;
  int before = __shfl(sum, src, WAVE_SIZE) - __shfl(n, src, WAVE_SIZE);
  for (int j0 = 0; j0 < per_lane; j0 += 64) {
    const int b = src * per_lane + j0 + lane;
    const int c = j0 + lane < per_lane && b < B
                      ? units_of(seq_lens[b], window, u) : 0;
    const int end = before + scan64(c);
    const unsigned long long hit = __ballot(end > begin);
    if (hit) {
      const int k = __ffsll(hit) - 1;
      *seq = src * per_lane + j0 + k;
      *at = begin - (__shfl(end, k, WAVE_SIZE) - __shfl(c, k, WAVE_SIZE));
      break;
    }
    before = __shfl(end, 63, WAVE_SIZE);
  }
  return min(per, total - begin);
}

// 16 bytes, or 2, of a lane to LDS
DEVINL void write16(uint32_t at, u32x4v v) {
  asm volatile("ds_write_b128 %0, %1" ::"v"(at), "v"(v) : "memory");
}
DEVINL void write2(uint32_t at, uint32_t v) {
  asm volatile("ds_write_b16 %0, %1" ::"v"(at), "v"(v) : "memory");
}

// Eight pairs of values turned, as rope_and_cache does it.
DEVINL void rotate8(u32x4v& a, u32x4v& b, const f32x4v (&c)[2],
                    const f32x4v (&s)[2]) {
  float x[8], y[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const float u = bf16_bits_to_f32((uint16_t)(a[r >> 1] >> (16 * (r & 1))));
    const float v = bf16_bits_to_f32((uint16_t)(b[r >> 1] >> (16 * (r & 1))));
    x[r] = fmaf(u, c[r >> 2][r & 3], -v * s[r >> 2][r & 3]);
    y[r] = fmaf(v, c[r >> 2][r & 3], u * s[r >> 2][r & 3]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[i] = pack_bf16(x[2 * i], x[2 * i + 1]);
    b[i] = pack_bf16(y[2 * i], y[2 * i + 1]);
  }
}

}  // namespace

// The step's token of every sequence, its last one, where it is not in the cache yet
// and queries and keys are not rotated: the key goes with the queries as one more of
// their 16 columns, whose sums nobody reads, and is turned with them; the wave whose
// tile ends the sequence puts it and the value into the tile behind the copies, and
// into the cache. No sequence may read another's. At most 15 query heads a
// key/value head. us, in a row of such pairs: rope_and_cache and this kernel apart /
// together: one sequence of 1,000, 14 heads over 2 x 64 9.8 / 8.9, 32 over 8 x 128 11.6 /
// 10.8; 32 of up to 300 11.0 / 8.9; 96 of up to 1,900 109 / 104; 128 of up to 4,000 261
// / 252; no pair of one to 128 sequences of up to 4,000 slower. The kernel alone, without
// a token, takes what it took before it knew of them: one sequence of 600, 32 over 8 x
// 128 7.15 and 7.15, 64 of 130, 64 over 8 x 128 6.79 and 6.74, one of 22,000, 64 over 8 x
// 64 18.3 and 18.3.
struct NewTokens {
  const uint16_t *k, *v;  // [B, Hk, D] rows at strides
  int64_t k_stride, v_stride;
  const int* positions;    // [B]
  const float* cos_sin;    // [.., D]
  const int64_t* slots;    // [B], below 0: none, the sequence is all in the cache
  uint16_t *k_out, *v_out;  // the cache
};
// nothing: 72 bytes less of arguments, 0.03 us of a launch on the host
struct NoTokens {};

template <int D, bool FP8, int W, bool NEW>
__global__ __launch_bounds__(W * 64, W > 4 ? 1 : 2) void paged_decode_kernel(
    uint16_t* __restrict__ out,         // [B, Hq, D]
    float* __restrict__ tmp_acc,        // [parts, Hq, D]; null: a workgroup a
    float* __restrict__ tmp_ml,         // [parts, Hq, 2]      sequence and head
    const uint16_t* __restrict__ q,     // [B, Hq, D] rows at q_stride
    const uint8_t* __restrict__ k_cache,  // [NB, Hk, BS, D] bf16 | fp8
    const uint8_t* __restrict__ v_cache,  // [NB, Hk, D, BS]
    const int* __restrict__ block_tables, const int* __restrict__ seq_lens,
    const int B, const int max_blocks, const int Hk, const int G,
    const int bs_shift, const int64_t q_stride, const float scale,
    const int window, const float softcap, const float* __restrict__ sinks,
    const float v_scale, const std::conditional_t<NEW, NewTokens, NoTokens> nt) {
  static_assert(!(NEW && FP8), "");
  constexpr int ES = FP8 ? 1 : 2;
  constexpr int RB = D * ES;             // bytes a K row
  constexpr int CPR = RB / 16;
  constexpr int VB = PD_KT * ES;         // bytes of a V row in a tile
  constexpr int TILE = PD_KT * RB;       // bytes of K, and of V, in a tile
  constexpr int NC = TILE / 1024;        // copies of K, and of V
  constexpr int KC = D / 32;
  constexpr int MT = D / 16;
  constexpr int U = W * PD_KT;           // tokens a unit
  constexpr int MROW = D + 4;            // floats a row where sums are added
  constexpr int MERGE = W * 16 * MROW * 4;
  constexpr int RING = W * 2 * TILE;
  constexpr int SMEM = MERGE > RING ? MERGE : RING;
  __shared__ __attribute__((aligned(1024))) uint8_t S[SMEM];
  __shared__ float ms[W][16], ls[W][16];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15;
  const int l4 = lane >> 4;
  const int hk = blockIdx.x;
  const int Hq = Hk * G;
  const int BS = 1 << bs_shift;

  // ---- this workgroup's run of units ---------------------------------------------
  int seq, at, todo, per = 1;  // sequence, unit of it, units left; of a full run
  if (tmp_acc == nullptr) {
    seq = blockIdx.y;
    at = 0;
    todo = units_of(seq_lens[seq], window, U);
    if (todo == 0)  // no tokens: zeros
      for (int e = tid; e < G * (D / 4); e += W * 64)
        *reinterpret_cast<uint2*>(out + ((size_t)seq * Hq + hk * G) * D + e * 4) =
            make_uint2(0, 0);
  } else {
    todo = find_run(seq_lens, window, U, B, blockIdx.y, gridDim.y, &seq, &at, &per);
  }
  int done = 0;  // units of the run so far
  seq = __builtin_amdgcn_readfirstlane(seq);
  at = __builtin_amdgcn_readfirstlane(at);
  todo = __builtin_amdgcn_readfirstlane(todo);

  uint8_t* Kt = S + wid * (2 * TILE);
  uint8_t* Vt = Kt + TILE;
  // ---- what a lane copies: byte offsets within a page ------------------------------
  // K: row lane / CPR of the copy's 64 / CPR rows; V: row lane / (VB / 16)
  const uint32_t k_row = lane / CPR;
  const uint32_t k_ch = (lane % CPR) ^ swz_k<CPR>(k_row);
  const uint32_t v_row = lane / (VB / 16);
  const uint32_t v_tok = ((lane % (VB / 16)) ^ swz_v<FP8>(v_row)) * (16 / ES);
  const bool v_second = v_tok >= (uint32_t)BS;  // of two pages of 16
  const uint32_t v_off = (v_row * BS + (v_tok & (BS - 1))) * ES;
  const int64_t page_bytes = (int64_t)Hk * BS * RB;
  const int64_t head_off = (int64_t)hk * BS * RB;
  // ---- what a lane reads ------------------------------------------------------------
  const int rr = 8 * (l15 >> 2) + (l15 & 3);
  const uint32_t k_at = lds_at(Kt) + rr * RB + (l4 ^ swz_k<CPR>(rr)) * 16;
  const uint32_t v_at =
      FP8 ? lds_at(Vt) + l15 * VB + ((l4 >> 1) ^ swz_v<FP8>(l15)) * 16 +
                (l4 & 1) * 8
          : lds_at(Vt) + l15 * VB + (l4 ^ swz_v<FP8>(l15)) * 16;

  while (todo > 0) {
    const int L = seq_lens[seq];
    int pos = 0;
    int64_t slot = -1;
    if constexpr (NEW) {  // asked for with L: one wait of the scalar unit
      pos = ((const __attribute__((address_space(4))) int*)nt.positions)[seq];
      slot = ((const __attribute__((address_space(4))) int64_t*)nt.slots)[seq];
      asm volatile("" ::"s"(L), "s"(pos), "s"(slot));
    }
    const int lo = window > 0 ? max(0, L - window) : 0;
    const int units = units_of(L, window, U);
    if (at >= units) {  // a sequence without tokens
      ++seq;
      at = 0;
      continue;
    }
    const int t0 = at, t1 = min(units, at + todo);
    if (tmp_acc != nullptr && t0 == 0 && hk == 0 && tid == 0)
      part_runs(tmp_ml, gridDim.y, B, Hq)[seq] =
          make_int2(blockIdx.y, blockIdx.y + (done + units - 1) / per);
    const int unit0 = lo / U;
    // constant memory: read by the scalar unit, no vector load among the copies
    const auto* btab = (const __attribute__((address_space(4))) int*)(
        block_tables + (size_t)seq * max_blocks);

    // ---- Q: B operands, head l15 -----------------------------------------------------
    bf16x8v qf[KC];
    {
      const uint16_t* row = q + (size_t)seq * q_stride +
                            (size_t)(hk * G + min(l15, G - 1)) * D;
      if constexpr (NEW)
        if (l15 == G) row = nt.k + (size_t)seq * nt.k_stride + hk * D;
#pragma unroll
      for (int s = 0; s < KC; ++s)
        qf[s] = *(const bf16x8v*)(row + (FP8 ? ((s >> 1) * 4 + l4) * 16 + (s & 1) * 8
                                             : s * 32 + l4 * 8));
    }
    // NEW: what they are turned by, and the new value
    f32x4v qc[KC / 2][2], qs[KC / 2][2];
    uint32_t v_new[D / 64];
    if constexpr (NEW) {
      const float* turn = nt.cos_sin + (size_t)pos * D;
      const uint16_t* vr = nt.v + (size_t)seq * nt.v_stride + hk * D;
#pragma unroll
      for (int i = 0; i < D / 64; ++i) v_new[i] = vr[i * 64 + lane];
#pragma unroll
      for (int s = 0; s < KC / 2; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          qc[s][i] = *(const f32x4v*)(turn + s * 32 + l4 * 8 + i * 4);
          qs[s][i] = *(const f32x4v*)(turn + D / 2 + s * 32 + l4 * 8 + i * 4);
        }
    }
    f32x4v o[MT] = {};
    float m = kLowest, l = 0.f;
    // above 0 also for a scale of 0: hidden scores are multiplied by it too
    const float c =
        softcap > 0.f ? 1.f : fmaxf(fabsf(scale) * kLog2e, 1e-20f);

    // this wave's tiles: from first on, a unit apart
    int first = (unit0 + t0) * U + wid * PD_KT;
    if (first + PD_KT <= lo) first += U;
    const int end = min(L, (unit0 + t1) * U);
    // past the end the copies are of the last tile again: the count of copies in
    // flight stays the same
    const int last = (L - 1) & ~(PD_KT - 1);
    auto pages = [&](int tok, int (&p)[2]) INL {  // of the tile's two halves
      const int at = min(tok, last);
      p[0] = btab[at >> bs_shift];
      p[1] = btab[min(bs_shift == 4 ? at + 16 : at, L - 1) >> bs_shift];
    };
    auto issue_k = [&](int tok, const int (&p)[2]) INL {
      const int64_t in = head_off + (int64_t)(min(tok, last) & (BS - 1)) * RB;
      const uint8_t* b0 = k_cache + p[0] * page_bytes + in;
      const uint8_t* b1 = k_cache + p[1] * page_bytes + in;
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        constexpr int RC = 64 / CPR;  // rows a copy
        const uint32_t off = k_row * RB + (k_ch ^ swz_k<CPR>(i * RC)) * 16;
        // the second 16 rows: of the second page, if pages have 16
        const uint8_t* b = i < NC / 2 ? b0 + i * 1024
                           : bs_shift == 4 ? b1 + (i - NC / 2) * 1024
                                           : b0 + i * 1024;
        copy16_to_lds(b + off, Kt + i * 1024);
      }
    };
    auto issue_v = [&](int tok, const int (&p)[2]) INL {
      const int64_t in = head_off + (int64_t)(min(tok, last) & (BS - 1)) * ES;
      const int64_t page = v_second ? p[1] : p[0];
      const uint8_t* b = v_cache + in + page * page_bytes + v_off;
#pragma unroll
      for (int i = 0; i < NC; ++i)
        copy16_to_lds(b + i * (1024 / VB) * BS * ES, Vt + i * 1024);
    };

    // NEW: the tile of this wave that the new token is put into
    const int fresh = NEW && slot >= 0 && last >= first && last < end &&
                              (last - first) % U == 0
                          ? last : -1;
    if (first < end) {
      int nx[2];
      pages(first, nx);
      issue_k(first, nx);
      issue_v(first, nx);
      pages(first + U, nx);
      if constexpr (NEW) {
        // What was asked for before K and V is here. Tied to it, or the compiler
        // moves the arithmetic ahead and has it wait for every copy.
        wait_copies<2 * NC>();
#pragma unroll
        for (int s = 0; s < KC; ++s) asm volatile("" : "+v"(qf[s]));
#pragma unroll
        for (int s = 0; s < KC / 2; ++s)
#pragma unroll
          for (int i = 0; i < 2; ++i)
            asm volatile("" : "+v"(qc[s][i]), "+v"(qs[s][i]));
#pragma unroll
        for (int s = 0; s < KC / 2; ++s) {
          u32x4v a = __builtin_bit_cast(u32x4v, qf[s]);
          u32x4v b = __builtin_bit_cast(u32x4v, qf[s + KC / 2]);
          rotate8(a, b, qc[s], qs[s]);
          qf[s] = __builtin_bit_cast(bf16x8v, a);
          qf[s + KC / 2] = __builtin_bit_cast(bf16x8v, b);
        }
      }
      // here, not at the end: the barriers of the sums wait for stores
      if constexpr (NEW) {
        if (fresh >= 0) {
          const int64_t row = (slot >> bs_shift) * Hk + hk;
          const int in = (int)(slot & (BS - 1));
          if (l15 == G) {
            uint16_t* dst = nt.k_out + (row * BS + in) * D + l4 * 8;
#pragma unroll
            for (int s = 0; s < KC; ++s)
              *reinterpret_cast<bf16x8v*>(dst + s * 32) = qf[s];
          }
#pragma unroll
          for (int i = 0; i < D / 64; ++i)
            nt.v_out[(row * D + i * 64 + lane) * BS + in] = (uint16_t)v_new[i];
        }
      }
      if (scale < 0.f && (!NEW || l15 < G)) {  // the sign goes with q, as c takes
#pragma unroll  // maxima; with copies on their way, because it waits for q
        for (int s = 0; s < KC; ++s)
          qf[s] = __builtin_bit_cast(
              bf16x8v, __builtin_bit_cast(u32x4v, qf[s]) ^ 0x80008000u);
      }
      for (int tok = first; tok < end; tok += U) {
        wait_copies<NC>();
        if (NEW && tok == fresh && l15 == G) {
          const int r = (L - 1) & (PD_KT - 1);
#pragma unroll
          for (int s = 0; s < KC; ++s)
            write16(lds_at(Kt) + r * RB + ((s * 4 + l4) ^ swz_k<CPR>(r)) * 16,
                    __builtin_bit_cast(u32x4v, qf[s]));
        }
        u32x4v kr[KC * ES];  // [chunk group][t]
        if constexpr (CPR == 16)
          read8<4 * RB>(kr, k_at, k_at ^ 64, k_at ^ 128, k_at ^ 192);
        else if constexpr (CPR == 8)
          read4<4 * RB>(kr, k_at, k_at ^ 64);
        else
          read2<4 * RB>(kr, k_at);
        issue_k(tok + U, nx);

        // token of s[t][r]: tok + 8 l4 + 4 t + r
        f32x4v s[2] = {};
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int k = 0; k < KC; ++k) {
            bf16x8v a;
            if constexpr (FP8) {
              const u32x4v r = kr[(k >> 1) * 2 + t];
              a = k & 1 ? widen(r[2], r[3]) : widen(r[0], r[1]);
            } else {
              a = __builtin_bit_cast(bf16x8v, kr[k * 2 + t]);
            }
            s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[k], s[t], 0, 0, 0);
          }
        if (softcap > 0.f) {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            s[e >> 2][e & 3] =
                softcap * tanhf(s[e >> 2][e & 3] * fabsf(scale) / softcap) * kLog2e;
        }
        const bool cut = tok + PD_KT > L;
        if (cut || tok < lo) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int k = tok + 8 * l4 + e;
            s[e >> 2][e & 3] = k >= lo && k < L ? s[e >> 2][e & 3] : kHidden;
          }
        }
        float mx = s[0][0];
#pragma unroll
        for (int e = 1; e < 8; ++e) mx = fmaxf(mx, s[e >> 2][e & 3]);
        mx = over_head(mx, [](float a, float b) { return fmaxf(a, b); }) * c;
        // rescaled when a maximum moved: its own weight is then 1, without error
        if (__any(mx > m)) {
          const float m2 = fmaxf(m, mx);
          const float f = __builtin_amdgcn_exp2f(m - m2);
          m = m2;
          l *= f;
#pragma unroll
          for (int t = 0; t < MT; ++t) o[t] *= f;
        }
        u32x4v pk;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const float p0 = __builtin_amdgcn_exp2f(fmaf(s[e >> 2][e & 3], c, -m));
          const float p1 =
              __builtin_amdgcn_exp2f(fmaf(s[e >> 2][(e & 3) + 1], c, -m));
          l += p0 + p1;
          pk[e >> 1] = pack_bf16(p0, p1);
        }

        wait_copies<NC>();
        if (NEW && tok == fresh) {
          const int r = (L - 1) & (PD_KT - 1);
#pragma unroll
          for (int i = 0; i < D / 64; ++i) {
            const int d = i * 64 + lane;
            write2(lds_at(Vt) + d * VB + ((r >> 3) ^ swz_v<FP8>(d)) * 16 + (r & 7) * 2,
                   v_new[i]);
          }
        }
        using VR = std::conditional_t<FP8, u32x2v, u32x4v>;
        VR vr[MT];
        read_rows(vr, v_at);
        issue_v(tok + U, nx);
        pages(tok + 2 * U, nx);
        // slots past the end may hold anything: weight 0 times it
        u32x4v keep = {~0u, ~0u, ~0u, ~0u};
        if (cut) {
          const int n = L - tok - 8 * l4;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            keep[i] = n >= 2 * i + 2 ? ~0u : n == 2 * i + 1 ? 0xffffu : 0u;
        }
        const bf16x8v pb = __builtin_bit_cast(bf16x8v, pk);
#pragma unroll
        for (int d = 0; d < MT; ++d) {
          u32x4v a;
          if constexpr (FP8)
            a = __builtin_bit_cast(u32x4v, widen(vr[d][0], vr[d][1]));
          else
            a = vr[d];
          if (cut) a &= keep;
          o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8v, a), pb, o[d], 0, 0, 0);
        }
      }
      wait_copies<0>();
    }

    // ---- the waves' sums ---------------------------------------------------------------
    l = over_head(l, [](float a, float b) { return a + b; });
    if (l4 == 0) {
      ms[wid][l15] = m;
      ls[wid][l15] = l;
    }
    __syncthreads();
    float M = kLowest;
#pragma unroll
    for (int w = 0; w < W; ++w) M = fmaxf(M, ms[w][l15]);
    const float f = __builtin_amdgcn_exp2f(m - M) * v_scale;
    float* sums = reinterpret_cast<float*>(S);
#pragma unroll
    for (int t = 0; t < MT; ++t)
      *reinterpret_cast<f32x4v*>(sums + (wid * 16 + l15) * MROW + t * 16 +
                                 l4 * 4) = o[t] * f;
    __syncthreads();
    const bool whole = t0 == 0 && t1 == units;
    const size_t part =
        whole ? seq : (size_t)blockIdx.y + seq;  // named by run + sequence
    for (int e = tid; e < G * (D / 4); e += W * 64) {
      const int g = e / (D / 4), d = e % (D / 4) * 4;
      float Mg = kLowest, lg = 0.f;
#pragma unroll
      for (int w = 0; w < W; ++w) Mg = fmaxf(Mg, ms[w][g]);
#pragma unroll
      for (int w = 0; w < W; ++w)
        lg += ls[w][g] * __builtin_amdgcn_exp2f(ms[w][g] - Mg);
      f32x4v s = {};
#pragma unroll
      for (int w = 0; w < W; ++w)
        s += *reinterpret_cast<const f32x4v*>(sums + (w * 16 + g) * MROW + d);
      const size_t row = part * Hq + hk * G + g;
      if (whole) {
        if (sinks != nullptr)
          lg += __builtin_amdgcn_exp2f(sinks[hk * G + g] * kLog2e - Mg);
        s *= 1.f / lg;
        *reinterpret_cast<uint2*>(out + row * D + d) =
            make_uint2(pack_bf16(s[0], s[1]), pack_bf16(s[2], s[3]));
      } else {
        *reinterpret_cast<f32x4v*>(tmp_acc + row * D + d) = s;
        if (d == 0) {
          tmp_ml[row * 2] = Mg;  // in units of log2
          tmp_ml[row * 2 + 1] = lg;
        }
      }
    }
    __syncthreads();
    todo -= t1 - t0;
    done += t1 - t0;
    ++seq;
    at = 0;
  }
}

// Adds up the parts of the sequences that several runs share: a workgroup a
// sequence and key/value head, groups of G D / 4 threads share the parts. What bounds it:
// one round trip after the other, for the sequence's runs, which its first run has left,
// for the maxima and sums, beside which a thread's first parts are on their way. us of it,
// the runs found from the lengths again and a round trip for each / so: 128 sequences of
// up to 4,096, 32 heads over 8 of 128 7.0 / 5.6; 200 of up to 3,001, 64 over 8 of 64 8.7 /
// 5.8; one of 32,000, 64 over 8 of 128 7.7 / 7.2. Eight parts ahead 6.2 for the two that
// most sequences have.
template <int D>
__global__ __launch_bounds__(256) void paged_decode_reduce_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ tmp_acc,
    const float* __restrict__ tmp_ml, const int* __restrict__ seq_lens,
    const float* __restrict__ sinks, const int B, const int Hk, const int G,
    const int window, const int u, const int runs) {
  const int seq = blockIdx.y, hk = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int Hq = Hk * G;
  const int2 range = part_runs(const_cast<float*>(tmp_ml), runs, B, Hq)[seq];
  if (units_of(seq_lens[seq], window, u) == 0) {  // no tokens: zeros
    for (int e = tid; e < G * (D / 4); e += 256)
      *reinterpret_cast<uint2*>(out + ((size_t)seq * Hq + hk * G) * D + e * 4) =
          make_uint2(0, 0);
    return;
  }
  const int r0 = range.x, r1 = range.y;
  if (r0 == r1) return;  // finished by its run

  extern __shared__ float wt[];  // [G][runs]
  __shared__ float den[16];
  __shared__ f32x4v sums[256];
  const int parts = r1 - r0 + 1;
  const size_t row0 = ((size_t)r0 + seq) * Hq + hk * G;
  const int per_part = G * (D / 4);
  const int groups = max(1, 256 / per_part);
  const int grp = tid / per_part;
  const int mine = groups > 1 ? grp : 0;
  constexpr int AHEAD = 4;
  f32x4v ahead[AHEAD];
  {
    const int e = min(groups > 1 ? tid % per_part : tid, per_part - 1);
    const float* src = tmp_acc + (row0 + e / (D / 4)) * D + e % (D / 4) * 4;
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)  // past the last one that one again
      ahead[i] = *reinterpret_cast<const f32x4v*>(
          src + (size_t)min(mine + i * groups, parts - 1) * Hq * D);
  }
  for (int g = tid >> 6; g < G; g += 4) {  // a wave a head
    const f32x2v* ml = reinterpret_cast<const f32x2v*>(tmp_ml) + row0 + g;
    const f32x2v first = ml[(size_t)min(lane, parts - 1) * Hq];
    float M = first[0], l = 0.f;
    for (int r = lane + 64; r < parts; r += 64) M = fmaxf(M, ml[(size_t)r * Hq][0]);
    M = wave_reduce_max(M);
    for (int r = lane; r < parts; r += 64) {
      const f32x2v v = r < 64 ? first : ml[(size_t)r * Hq];
      const float w = __builtin_amdgcn_exp2f(v[0] - M);
      l += v[1] * w;
      wt[g * runs + r] = w;
    }
    l = wave_reduce_sum(l);
    if (lane == 0)
      den[g] = l + (sinks != nullptr ? __builtin_amdgcn_exp2f(
                                           sinks[hk * G + g] * kLog2e - M)
                                     : 0.f);
  }
  __syncthreads();
  for (int e0 = 0; e0 < per_part; e0 += 256) {
    const int e = groups > 1 ? tid % per_part : e0 + tid;
    const bool on = e < per_part && grp < groups;
    const int g = e / (D / 4), d = e % (D / 4) * 4;
    f32x4v s = {};
    if (on) {
      const float* src = tmp_acc + (row0 + g) * D + d;
      int r = mine;
      if (e0 == 0)
#pragma unroll
        for (int i = 0; i < AHEAD; ++i, r += groups)
          if (r < parts) s += ahead[i] * wt[g * runs + r];
#pragma unroll 8
      for (; r < parts; r += groups)
        s += *reinterpret_cast<const f32x4v*>(src + (size_t)r * Hq * D) * wt[g * runs + r];
    }
    if (groups > 1) {
      sums[tid] = s;
      __syncthreads();
      if (grp > 0) return;
      for (int k = 1; k < groups; ++k) s += sums[k * per_part + e];
    }
    if (!on) continue;
    s *= 1.f / den[g];
    *reinterpret_cast<uint2*>(out + ((size_t)seq * Hq + hk * G + g) * D + d) =
        make_uint2(pack_bf16(s[0], s[1]), pack_bf16(s[2], s[3]));
  }
}

// Runs the units are dealt to; 0: every sequence and head has a workgroup of its
// own and no second kernel. us without / with runs: one sequence, 8 heads x 128, of
// 600 7.6 / 13, of 1,000 9.4 / 13, of 4,000 25 / 13; 32 of 1,000 21 / 27; many
// sequences balance by themselves, 512 x 2 heads of 1,100 23 / 37, 96 x 8 of 3,000
// 154 / 146, but one long one among them would be waited for: up to 2,048 tokens.
// One run a CU, two with 64-wide heads, whose tiles are smaller: 200 x 8 heads of
// 3,001 in fp8 106 / 87 us with one / two; 96 x 8 x 128 144 / 149.
extern "C" int paged_decode_runs(int B, int Hk, int D, int max_len, int window) {
  const int n = window > 0 && window < max_len ? window : max_len;
  if (n <= 1024 || (n <= 2048 && B * Hk >= 768)) return 0;
  return clamp_int((D == 128 ? 256 : 512) / Hk, 1, PD_MAX_RUNS);
}

// new_k null: every token is in the cache, q is rotated
extern "C" void launch_paged_decode(
    void* out, const void* q, void* k_cache, void* v_cache,
    const int* block_tables, const int* seq_lens, int B, int Hq, int Hk, int D,
    int BS, int max_blocks, int64_t q_stride, float scale, int window,
    float softcap, const float* sinks, int runs, float* tmp_acc, float* tmp_ml,
    bool kv_fp8, float k_scale, float v_scale, const void* new_k, const void* new_v,
    int64_t k_stride, int64_t v_stride, const int* positions, const float* cos_sin,
    const int64_t* slots, hipStream_t stream, bool* launched) {
  const int G = Hq / Hk;
  *launched = false;
  if (G > 16 || (D != 64 && D != 128) || (new_k != nullptr && (kv_fp8 || G > 15)))
    return;
  if (BS != 16 && BS != 32 && BS != 64) return;
  *launched = true;
  const int shift = __builtin_ctz(BS);
  const dim3 grid(Hk, runs > 0 ? runs : B);
  auto run = [&](auto kernel, int waves, auto tokens) {
    kernel<<<grid, waves * 64, 0, stream>>>(
        (uint16_t*)out, tmp_acc, tmp_ml, (const uint16_t*)q,
        (const uint8_t*)k_cache, (const uint8_t*)v_cache, block_tables, seq_lens,
        B, max_blocks, Hk, G, shift, q_stride,
        kv_fp8 ? scale * k_scale : scale, window, softcap, sinks,
        kv_fp8 ? v_scale : 1.f, tokens);
  };
  // few workgroups: more waves each (one sequence, 8 heads x 128, of 1,000: 4 waves
  // 10.1 us, 8 9.4; 512 workgroups of 200 tokens: 4 waves 12 us, 8 24)
  const bool wide = runs == 0 && B * Hk <= 256;
  auto pick = [&](auto tokens) {
    constexpr bool N = std::is_same_v<decltype(tokens), NewTokens>;
    if (D == 128) wide ? run(paged_decode_kernel<128, false, 8, N>, 8, tokens)
                       : run(paged_decode_kernel<128, false, 4, N>, 4, tokens);
    else wide ? run(paged_decode_kernel<64, false, 16, N>, 16, tokens)
              : run(paged_decode_kernel<64, false, 4, N>, 4, tokens);
  };
  const NoTokens none{};
  if (new_k != nullptr) {
    pick(NewTokens{(const uint16_t*)new_k, (const uint16_t*)new_v, k_stride, v_stride,
                   positions, cos_sin, slots, (uint16_t*)k_cache,
                   (uint16_t*)v_cache});
  } else if (!kv_fp8) {
    pick(none);
  } else if (D == 128) {
    wide ? run(paged_decode_kernel<128, true, 16, false>, 16, none)
         : run(paged_decode_kernel<128, true, 4, false>, 4, none);
  } else {
    wide ? run(paged_decode_kernel<64, true, 16, false>, 16, none)
         : run(paged_decode_kernel<64, true, 4, false>, 4, none);
  }
  if (runs > 0) {
    auto reduce = [&](auto kernel) {
      kernel<<<dim3(Hk, B), 256, G * runs * sizeof(float), stream>>>(
          (uint16_t*)out, tmp_acc, tmp_ml, seq_lens, sinks, B, Hk, G, window, 4 * PD_KT,
          runs);
    };
    if (D == 128) reduce(paged_decode_reduce_kernel<128>);
    else reduce(paged_decode_reduce_kernel<64>);
  }
}
