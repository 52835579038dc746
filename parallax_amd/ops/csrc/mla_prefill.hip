// MLA prefill for gfx950: prompt portions of requests against their contexts.
//
//   mla_expand   keys k = latent . W_uk[h]^T and values v = latent . W_uv[h]^T of
//                a run of context rows, for every head, to bf16 pairs (below)
//   mla_prefill  flash attention of the portion's rows over those keys and the
//                rotated key parts, which are read from the context rows
//
// Between the bf16 inputs (queries, rotated parts, latents, weights) and the bf16
// result a value that is not a bf16 number (k, v, the softmax weights p) enters
// the matrix instructions as hi + lo, hi = bf16(x), lo = bf16(x - hi), 16 to 17
// bits of mantissa where fp32 has 24; q . k takes two products, p . v three (lo .
// lo is 2^-18 of it). The sums are fp32. It is the rounded result that is as exact
// as with fp32 products, whose own error is 1e-6 of it: against 64 bits (8 to 128
// heads, 40 to 2,500 rows, contexts to 9,000, queries to 4 times as large) 0.001649
// to 0.001665 either way, the same to the fifth digit; 0.4% of the values round to
// the neighbouring bf16 number.
//
// Why keys are expanded: per pair of row and key a head then takes 320 + 384
// multiply-adds (the parts counted); in latent space 1,088 + 1,024. A run is at most
// 2^20 / heads context rows, 1 GB of parts at any number of heads (the caller's
// rule); longer contexts go run by run, the fp32 state of the rows in memory between.
//
// What bounds it: matrix cores, 44 instructions of 32x32x16 per wave and 32 keys
// beside about 900 VALU cycles; two workgroups a CU overlap them. A prompt of
// 2,500 rows at 128 heads: expansion 230 us, attention 500 us; the fp32 torch
// operations in latent space that this replaced 25 ms. 512 rows on a context of
// 40,000: 8.2 ms, before 71 ms.

#include <type_traits>

#include "common.h"

#define MP_R 512    // latent rank
#define MP_DR 64    // rotated part
#define MP_DK 576   // values a context row
#define MP_D 128    // key and value width a head
#define MP_ROWS 128 // query rows a workgroup
#define MP_KT 32    // keys a tile

typedef float f32x16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2n __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4v __attribute__((ext_vector_type(4)));

namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kHidden = -__builtin_inff();  // score of a key that is not seen
constexpr float kLowest = -1e30f;              // where a maximum starts

DEVINL uint32_t pack_bf16(float a, float b) {
  bf16x2n p;
  p[0] = (__bf16)a;
  p[1] = (__bf16)b;
  return __builtin_bit_cast(uint32_t, p);
}

// two fp32 values to their hi and lo parts
DEVINL void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  hi = pack_bf16(a, b);
  lo = pack_bf16(a - __uint_as_float(hi << 16),
                 b - __uint_as_float(hi & 0xffff0000u));
}

DEVINL void copy16_to_lds(const void* src, void* dst) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)src,
      (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

DEVINL float max_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

DEVINL float sum_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

}  // namespace

// Portions of several requests in one pair of launches, whose contexts are read from the
// cache's pages: a launch more for each, a copy of its rows and a conversion of its pages'
// numbers cost more than a short portion's work, and leave most of the chip idle. us of
// whole layers of 128 heads, a request at a time / so: three of 572 rows together 886 / 842,
// in fp8 of 200 together 413 / 373, two of 2,500 together 2,957 / 2,903, one of 1,365
// 1,679 / 1,664.
#define MP_MAX_PORTIONS 16
struct Portion {
  int q0, T;     // query rows
  int n, base;   // context rows, and where theirs begin among the expanded ones
  int tile;      // first tile of MP_ROWS query rows
  int seq;       // row of the block tables
};
struct Portions {
  Portion p[MP_MAX_PORTIONS];
  int count;
};
struct Pages {
  const uint16_t* cache;  // [NB, 1 << shift, 576]
  const int* tables;      // [B, max_blocks]
  int max_blocks, shift;
  uint16_t* pe;           // rotated parts of the expanded rows [.., 64], written
};
struct NoPages {};

// ---- keys and values of a run ------------------------------------------------------
// 128 context rows x 128 features a workgroup, 4 waves of 64 x 64, both operands
// global -> LDS directly, 128 bytes of every row a stage. Keys come out as
// [head, row, feature] and values as [head, feature, row]: the operand order is
// swapped between the two, so that a lane's four neighbouring registers are
// neighbours in memory either way. Rows past the run are written as zeros.
// What bounds it: LDS reads, as long as products and stages that it waits for beside
// them. 1,900 rows, 128 heads: 128 us; stored from the accumulators, 16 bytes of 32 rows
// an instruction, 155; five stages of 64 bytes in a ring 141.

template <bool PAGED>
__global__ __launch_bounds__(256, 2) void mla_expand_kernel(
    uint16_t* __restrict__ k_hi, uint16_t* __restrict__ k_lo,  // [H, cap, 128]
    uint16_t* __restrict__ v_hi, uint16_t* __restrict__ v_lo,  // [H, 128, cap]
    const uint16_t* __restrict__ rows,  // [n, 576], not PAGED
    const uint16_t* __restrict__ w_uk,  // [H, 128, 512]
    const uint16_t* __restrict__ w_uv, int n, const int cap,
    const std::conditional_t<PAGED, Portions, NoPages> portions,
    const std::conditional_t<PAGED, Pages, NoPages> pages) {
  constexpr int BKB = 128;
  __shared__ __attribute__((aligned(16))) uint8_t S0[256 * BKB];
  __shared__ __attribute__((aligned(16))) uint8_t S1[256 * BKB];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, l31 = lane & 31;
  int r0 = blockIdx.y * 128;  // of the context; at0: of the expanded rows
  const int at0 = r0;
  const int h = blockIdx.x >> 1;
  const bool val = blockIdx.x & 1;
  const int* btab = nullptr;
  if constexpr (PAGED) {
    int i = portions.count - 1;
    while (i > 0 && portions.p[i].base > at0) --i;
    n = portions.p[i].n;
    r0 = at0 - portions.p[i].base;
    btab = pages.tables + (size_t)portions.p[i].seq * pages.max_blocks;
  }
  auto context_row = [&](int r) {
    if constexpr (PAGED) {
      const int slot = r & ((1 << pages.shift) - 1);
      return pages.cache +
             (((size_t)btab[r >> pages.shift] << pages.shift) + slot) * MP_DK;
    } else {
      return rows + (size_t)r * MP_DK;
    }
  };
  const uint8_t* w =
      (const uint8_t*)((val ? w_uv : w_uk) + (size_t)h * MP_D * MP_R);

  // a thread's chunk of rows tid / 8 + 32 i: weights are LDS rows 0..127
  const int src = ((tid & 7) ^ ((tid >> 4) & 7)) * 16;
  const uint8_t *wp[4], *rp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = i * 32 + (tid >> 3);
    wp[i] = w + (size_t)r * (MP_R * 2) + src;
    rp[i] = (const uint8_t*)context_row(min(r0 + r, n - 1)) + src;
  }
  if constexpr (PAGED) {  // eight threads a row
    if (blockIdx.x == 0)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<u32x4v*>(pages.pe + (size_t)(at0 + i * 32 + (tid >> 3)) * MP_DR +
                                   (tid & 7) * 8) =
            *reinterpret_cast<const u32x4v*>((const uint16_t*)(rp[i] - src) + MP_R +
                                             (tid & 7) * 8);
  }
  auto issue = [&](int kt, uint8_t* S) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      copy16_to_lds(wp[i] + kt * BKB, S + (i * 32 + wid * 8) * BKB);
      copy16_to_lds(rp[i] + kt * BKB, S + (128 + i * 32 + wid * 8) * BKB);
    }
  };
  // registers run over the features of a key, over the rows of a value
  const int ra = (val ? 128 : 0) + (wid & 1) * 64;
  const int rb = (val ? 0 : 128) + (wid >> 1) * 64;
  const int swz_l = (l31 >> 1) & 7;
  f32x16v acc[2][2] = {};
  auto stage = [&](const uint8_t* S) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int c = ((2 * ks + half) ^ swz_l) * 16;
      bf16x8v a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[i] = *(const bf16x8v*)(S + (ra + i * 32 + l31) * BKB + c);
        b[i] = *(const bf16x8v*)(S + (rb + i * 32 + l31) * BKB + c);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j],
                                                              acc[i][j], 0, 0, 0);
    }
  };
  constexpr int NK = MP_R * 2 / BKB;
  issue(0, S0);
#pragma unroll
  for (int kt = 0; kt < NK; kt += 2) {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __syncthreads();
    issue(kt + 1, S1);
    stage(S0);
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    if (kt + 2 < NK) issue(kt + 2, S0);
    stage(S1);
  }

  // Through LDS, so that a wave stores whole lines: rows of 128 (of a key's features, or
  // of one feature's context rows), 16-byte chunk c of row r at c ^ (r & 15).
  __syncthreads();  // every wave is done with the stages
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = (rb & 127) + j * 32 + l31;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = (ra & 127) + i * 32 + 8 * q + 4 * half;
        uint2 a, b;
        float x[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int tok = r0 + (val ? row + s : col);
          x[s] = tok < n ? acc[i][j][4 * q + s] : 0.f;
        }
        split2(x[0], x[1], a.x, b.x);
        split2(x[2], x[3], a.y, b.y);
        const int at = col * 256 + ((row >> 3) ^ (col & 15)) * 16 + half * 8;
        *reinterpret_cast<uint2*>(S0 + at) = a;
        *reinterpret_cast<uint2*>(S1 + at) = b;
      }
  }
  __syncthreads();
  const size_t base = (size_t)h * cap * MP_D + (val ? (size_t)at0 : (size_t)at0 * MP_D);
  const size_t pitch = val ? cap : MP_D;
  uint16_t* hi = (val ? v_hi : k_hi) + base;
  uint16_t* lo = (val ? v_lo : k_lo) + base;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = i * 16 + (tid >> 4), ch = tid & 15;
    const int at = row * 256 + (ch ^ (row & 15)) * 16;
    *reinterpret_cast<u32x4v*>(hi + row * pitch + ch * 8) =
        *reinterpret_cast<const u32x4v*>(S0 + at);
    *reinterpret_cast<u32x4v*>(lo + row * pitch + ch * 8) =
        *reinterpret_cast<const u32x4v*>(S1 + at);
  }
}

// ---- attention ------------------------------------------------------------------------
// 128 query rows of one head a workgroup, 32 a wave; see prefill_attention for
// the operand orders (S^T = K Q^T, O^T = V^T P, P from the accumulators).

template <bool PAGED>
__global__ __launch_bounds__(256, 2) void mla_prefill_kernel(
    uint16_t* __restrict__ out,           // [T, H, 128]
    float* __restrict__ state,            // [T, H, 130] or null
    const uint16_t* __restrict__ q_nope,  // [T, H, 128] by strides
    const uint16_t* __restrict__ q_pe,    // [T, H, 64]
    const uint16_t* __restrict__ k_hi, const uint16_t* __restrict__ k_lo,
    const uint16_t* __restrict__ v_hi, const uint16_t* __restrict__ v_lo,
    const uint16_t* __restrict__ rows,    // [n, 576]; PAGED: rotated parts [cap, 64]
    int T, const int H, int n, const int cap, int prefix,
    const int first_key, const int64_t q_row, const int64_t q_head,
    const float scale, const int first, const int last,
    const std::conditional_t<PAGED, Portions, NoPages> portions) {
  __shared__ __attribute__((aligned(16))) uint16_t Kh0[MP_KT * 128], Kl0[MP_KT * 128];
  __shared__ __attribute__((aligned(16))) uint16_t Kh1[MP_KT * 128], Kl1[MP_KT * 128];
  __shared__ __attribute__((aligned(16))) uint16_t R0[MP_KT * 64], R1[MP_KT * 64];
  __shared__ __attribute__((aligned(16))) uint16_t Vh0[MP_KT * 128], Vl0[MP_KT * 128];
  __shared__ __attribute__((aligned(16))) uint16_t Vh1[MP_KT * 128], Vl1[MP_KT * 128];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, l31 = lane & 31;
  // heads fastest: with 8 | H a head's blocks share an XCD's L2; the last rows
  // see the most keys and come first
  const int h = blockIdx.x % H;
  int tile = gridDim.x / H - 1 - blockIdx.x / H;
  int base = 0;
  if constexpr (PAGED) {
    int i = portions.count - 1;
    while (i > 0 && portions.p[i].tile > tile) --i;
    const Portion p = portions.p[i];
    tile -= p.tile;
    T = p.T;
    n = p.n;
    prefix = n - T;
    base = p.base;
    out += (size_t)p.q0 * H * MP_D;
    q_nope += p.q0 * q_row;
    q_pe += (size_t)p.q0 * H * MP_DR;
    rows += (size_t)base * MP_DR;
  }
  const int w0 = tile * MP_ROWS + wid * 32;
  const int row = w0 + l31;
  const bool row_ok = row < T;
  const int row_c = min(row, T - 1);
  // positions within this run of keys
  const int qpos = prefix + row - first_key;
  const int wpos_lo = prefix + w0 - first_key;
  const bool wave_on = w0 < T;
  const int wpos_hi = prefix + min(w0 + 31, T - 1) - first_key;
  const int pos_hi =
      prefix + min(tile * MP_ROWS + MP_ROWS - 1, T - 1) - first_key;
  const int kt_end = max(0, (min(n, pos_hi + 1) + MP_KT - 1) / MP_KT);

  bf16x8v qf[12];
  {
    const uint16_t* a =
        q_nope + (size_t)row_c * q_row + (size_t)h * q_head + half * 8;
    const uint16_t* b = q_pe + ((size_t)row_c * H + h) * MP_DR + half * 8;
#pragma unroll
    for (int s = 0; s < 12; ++s)
      qf[s] = s < 8 ? *(const bf16x8v*)(a + s * 16)
                    : *(const bf16x8v*)(b + (s - 8) * 16);
    if (scale < 0.f) {  // the sign goes with q: c takes maxima
#pragma unroll
      for (int s = 0; s < 12; ++s)
        qf[s] = __builtin_bit_cast(
            bf16x8v, __builtin_bit_cast(u32x4v, qf[s]) ^ 0x80008000u);
    }
  }
  f32x16v o[4] = {};
  float m = kLowest, l = 0.f;  // l: this half's keys only
  float* st = state + ((size_t)row_c * H + h) * 130;
  if (!first) {
    m = st[128];
    l = half == 0 ? st[129] : 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          o[t][4 * i + r] = st[t * 32 + 8 * i + 4 * half + r];
  }
  // above 0 also for a scale of 0: hidden scores are multiplied by it too
  const float c = fmaxf(fabsf(scale) * kLog2e, 1e-20f);

  // ---- copies: chunk numbers within a tile, LDS places XOR-swizzled by row ---------
  const uint16_t* kh = k_hi + ((size_t)h * cap + base) * MP_D;
  const uint16_t* kl = k_lo + ((size_t)h * cap + base) * MP_D;
  const uint16_t* vh = v_hi + (size_t)h * cap * MP_D + base;
  const uint16_t* vl = v_lo + (size_t)h * cap * MP_D + base;
  int k_at[2], v_at[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int ch = (wid * 2 + i) * 64 + lane;
    const int kr = ch >> 4, vr = ch >> 2;
    k_at[i] = kr * MP_D + ((ch & 15) ^ (kr & 15)) * 8;
    v_at[i] = vr * cap + ((ch & 3) ^ ((vr >> 2) & 3)) * 8;
  }
  const int pe_row = tid >> 3;
  constexpr int PE_ROW = PAGED ? MP_DR : MP_DK;
  const int pe_at = (PAGED ? 0 : MP_R) + ((tid & 7) ^ ((pe_row >> 1) & 7)) * 8;
  auto issue = [&](int kt, uint16_t* Kh, uint16_t* Kl, uint16_t* R,
                   uint16_t* Vh, uint16_t* Vl) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int dst = (wid * 2 + i) * 512;
      copy16_to_lds(kh + (size_t)kt * (MP_KT * MP_D) + k_at[i], Kh + dst);
      copy16_to_lds(kl + (size_t)kt * (MP_KT * MP_D) + k_at[i], Kl + dst);
      copy16_to_lds(vh + (size_t)kt * MP_KT + v_at[i], Vh + dst);
      copy16_to_lds(vl + (size_t)kt * MP_KT + v_at[i], Vl + dst);
    }
    copy16_to_lds(
        rows + (size_t)min(kt * MP_KT + pe_row, n - 1) * PE_ROW + pe_at,
        R + wid * 512);
  };

  // K row with bits 2 and 3 swapped: a lane half's weights are 8 neighbouring keys
  const int krow = (l31 & 0x13) | ((l31 & 4) << 1) | ((l31 & 8) >> 1);
  auto compute = [&](int kt, const uint16_t* Kh, const uint16_t* Kl,
                     const uint16_t* R, const uint16_t* Vh, const uint16_t* Vl)
      __attribute__((always_inline)) {
    const int kbase = kt * MP_KT;
    if (!wave_on || kbase > wpos_hi) return;
    f32x16v s = {}, s2 = {};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const int at = krow * 128 + ((2 * ks + half) ^ (krow & 15)) * 8;
      const bf16x8v a = *(const bf16x8v*)(Kh + at);
      const bf16x8v b = *(const bf16x8v*)(Kl + at);
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qf[ks], s, 0, 0, 0);
      s2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, qf[ks], s2, 0, 0, 0);
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const bf16x8v a = *(const bf16x8v*)(
          R + krow * 64 + ((2 * ks + half) ^ ((krow >> 1) & 7)) * 8);
      f32x16v& d = ks & 1 ? s2 : s;
      d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qf[8 + ks], d, 0, 0, 0);
    }
    s += s2;

    if (kbase + MP_KT - 1 > wpos_lo || kbase + MP_KT > n) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = kbase + 16 * (r >> 3) + 8 * half + (r & 7);
        s[r] = key <= qpos && key < n ? s[r] : kHidden;
      }
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = max_halves(mx) * c;
    // rescaled only when a maximum moved by more than 2^8
    if (__any(mx > m + 8.f)) {
      const float m2 = fmaxf(m, mx);
      const float f = __builtin_amdgcn_exp2f(m - m2);
      m = m2;
      l *= f;
#pragma unroll
      for (int t = 0; t < 4; ++t) o[t] *= f;
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      float p[8];
      u32x4v ph, pl;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        p[j] = __builtin_amdgcn_exp2f(fmaf(s[ks * 8 + j], c, -m));
        l += p[j];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t hi, lo;
        split2(p[2 * j], p[2 * j + 1], hi, lo);
        ph[j] = hi;
        pl[j] = lo;
      }
      const bf16x8v bh = __builtin_bit_cast(bf16x8v, ph);
      const bf16x8v bl = __builtin_bit_cast(bf16x8v, pl);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int d = t * 32 + l31;
        const int at = d * MP_KT + ((2 * ks + half) ^ ((d >> 2) & 3)) * 8;
        const bf16x8v ah = *(const bf16x8v*)(Vh + at);
        const bf16x8v al = *(const bf16x8v*)(Vl + at);
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, o[t], 0, 0, 0);
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl, o[t], 0, 0, 0);
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh, o[t], 0, 0, 0);
      }
    }
  };

  if (kt_end > 0) issue(0, Kh0, Kl0, R0, Vh0, Vl0);
  for (int kt = 0; kt < kt_end; kt += 2) {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __syncthreads();
    if (kt + 1 < kt_end) issue(kt + 1, Kh1, Kl1, R1, Vh1, Vl1);
    compute(kt, Kh0, Kl0, R0, Vh0, Vl0);
    if (kt + 1 >= kt_end) break;
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    if (kt + 2 < kt_end) issue(kt + 2, Kh0, Kl0, R0, Vh0, Vl0);
    compute(kt + 1, Kh1, Kl1, R1, Vh1, Vl1);
  }

  if (!row_ok) return;
  l = sum_halves(l);
  if (!last) {
    if (half == 0) {
      st[128] = m;
      st[129] = l;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          st[t * 32 + 8 * i + 4 * half + r] = o[t][4 * i + r];
    return;
  }
  const float inv = 1.f / l;
  uint16_t* dst = out + ((size_t)row * H + h) * MP_D + 4 * half;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint2 v;
      v.x = pack_bf16(o[t][4 * i] * inv, o[t][4 * i + 1] * inv);
      v.y = pack_bf16(o[t][4 * i + 2] * inv, o[t][4 * i + 3] * inv);
      *reinterpret_cast<uint2*>(dst + t * 32 + 8 * i) = v;
    }
}

extern "C" void launch_mla_prefill_run(
    void* out, float* state, const void* q_nope, const void* q_pe, void* k_hi,
    void* k_lo, void* v_hi, void* v_lo, const void* rows, const void* w_uk,
    const void* w_uv, int T, int H, int n, int cap, int prefix, int first_key,
    int64_t q_row, int64_t q_head, float scale, bool first, bool last,
    hipStream_t stream) {
  mla_expand_kernel<false><<<dim3(2 * H, ceil_div(n, 128), 1), 256, 0, stream>>>(
      (uint16_t*)k_hi, (uint16_t*)k_lo, (uint16_t*)v_hi, (uint16_t*)v_lo,
      (const uint16_t*)rows, (const uint16_t*)w_uk, (const uint16_t*)w_uv, n,
      cap, NoPages{}, NoPages{});
  mla_prefill_kernel<false><<<ceil_div(T, MP_ROWS) * H, 256, 0, stream>>>(
      (uint16_t*)out, state, (const uint16_t*)q_nope, (const uint16_t*)q_pe,
      (const uint16_t*)k_hi, (const uint16_t*)k_lo, (const uint16_t*)v_hi,
      (const uint16_t*)v_lo, (const uint16_t*)rows, T, H, n, cap, prefix,
      first_key, q_row, q_head, scale, first, last, NoPages{});
}

extern "C" int mla_prefill_max_portions() { return MP_MAX_PORTIONS; }

// lens: rows and context rows of each of count portions, starts: their first query row
// and their row of the block tables, in the order of their context rows, so that the
// longest tiles, which are dealt from the end, come first. cap: the sum of the contexts,
// each in multiples of 128.
extern "C" void launch_mla_prefill_paged(
    void* out, const void* q_nope, const void* q_pe, void* k_hi, void* k_lo, void* v_hi,
    void* v_lo, void* pe, const void* cache, const int* tables, int max_blocks, int shift,
    const void* w_uk, const void* w_uv, const int* lens, const int* starts, int count,
    int H, int cap, int64_t q_row, int64_t q_head, float scale, hipStream_t stream) {
  Portions ps{};
  ps.count = count;
  int base = 0, tiles = 0;
  for (int i = 0; i < count; ++i) {
    ps.p[i] = {starts[2 * i], lens[2 * i], lens[2 * i + 1], base, tiles,
               starts[2 * i + 1]};
    base += ceil_div(lens[2 * i + 1], 128) * 128;
    tiles += ceil_div(lens[2 * i], MP_ROWS);
  }
  mla_expand_kernel<true><<<dim3(2 * H, cap / 128, 1), 256, 0, stream>>>(
      (uint16_t*)k_hi, (uint16_t*)k_lo, (uint16_t*)v_hi, (uint16_t*)v_lo, nullptr,
      (const uint16_t*)w_uk, (const uint16_t*)w_uv, 0, cap, ps,
      Pages{(const uint16_t*)cache, tables, max_blocks, shift, (uint16_t*)pe});
  mla_prefill_kernel<true><<<tiles * H, 256, 0, stream>>>(
      (uint16_t*)out, nullptr, (const uint16_t*)q_nope, (const uint16_t*)q_pe,
      (const uint16_t*)k_hi, (const uint16_t*)k_lo, (const uint16_t*)v_hi,
      (const uint16_t*)v_lo, (const uint16_t*)pe, 0, H, 0, cap, 0, 0, q_row, q_head,
      scale, 1, 1, ps);
}
