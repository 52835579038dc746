// Varlen prefill attention over the paged KV cache for gfx950.
//
// A workgroup takes 128 (row, head) items of one request and one key/value
// head: item m is query row m / G of head m % G of the group, so the heads
// that share K and V share their tiles, and any group size and portion length
// fills the 32-item columns of a wave. Keys go by in tiles of 64:
//   S^T[64 x 32 items] = K . Q^T      mfma_f32_32x32x16_bf16, Q in registers
//   online softmax per item           one column = lanes l and l + 32
//   O^T[D x 32 items] += V^T . P      P straight from the registers of S^T
// An accumulator of S^T holds rows {4h + 8i + (0..3)} in lane half h. The rows
// of the K operand are taken in the order that swaps bits 2 and 3 of the row
// number, so that a half holds eight neighbouring tokens: exactly a B operand
// of the second product. P never touches LDS and a wave's softmax needs no
// other wave, which leaves one barrier a tile.
//
// bf16 tiles are copied global -> LDS directly (16 bytes a lane), a turn before
// their use; an fp8 cache passes through registers, where it is widened. 16-byte
// chunks are placed XOR-swizzled by row: a quarter wave reads 16 rows of one chunk
// column from 16 different bank groups.
//
// A turn takes the scores of one tile and the values of the tile before, whose
// weights depend on nothing of this turn. For 128-wide heads the two are interleaved
// by hand, matrix instruction by matrix instruction, where no mask cuts the tile: two
// waves a SIMD (240 registers) keep the matrix cores busy for 53% of the cycles
// instead of 40. For 64-wide heads, where softmax outweighs the products, a second
// set of scores costs the third wave a SIMD, and the turn goes through the two one
// after the other (interleaved 255 us for 4,500 rows of 64 heads over 8, apart 254;
// 3,000 rows with a window of 128 35.5 and 30).
//
// What bounds it: the card's power, and within a cycle how little the units overlap. The
// case below takes 5.53 M cycles of a CU, of which the matrix cores are busy for 53% and
// VALU instructions, four cycles each, would take 37. With operands of zeros the same
// products take 5.17 M (the accumulators are not rescaled), but at 2.38 GHz instead of
// 1.55 to 1.84: 2.17 ms for 3.0 to 3.5 (profiles/rocprof/prefill_attention_power.txt). The
// accumulators are rescaled only when an item's maximum moved, the mask is applied only in
// tiles that the diagonal, the window or the end of the sequence cuts.
//
// Measured (MI355X, bf16, 32 heads over 8 of 128, 8192 rows in two portions on
// prefixes of up to 20,000): 3.00 ms = 890 TFLOP/s of what the mask leaves; scores and
// values of one tile in turn, with a branch and a wait at every operand of V, 3.47. 5,700
// rows on an fp8 cache 425 to 338 us (conversions by the hardware's rounding), 64-wide
// heads 340 to 274; 8,192 rows without a prefix 228 to 213.

#include <type_traits>

#include "common.h"

#define PF_THREADS 256
#define PF_ITEMS 128  // (row, head) items a workgroup: 4 waves x 32
#define PF_KT 64      // keys a tile

typedef float f32x16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2n __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4v __attribute__((ext_vector_type(4)));

namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
// Score of a key that is not seen, and where an item's maximum starts. A tile in
// which an item sees nothing (a window, a split at the diagonal) leaves its m, l
// and O alone: -inf raises no maximum and weighs exp2(-inf) = 0. A finite hidden
// score would be rounded once in m and not in the weight's fma, whose exponent is
// then the rounding error: +8e20 for 64-wide heads.
constexpr float kHidden = -__builtin_inff();
constexpr float kLowest = -1e30f;

DEVINL float max_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v),
                                                  __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

DEVINL float sum_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v),
                                                  __float_as_uint(v), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

DEVINL uint32_t pack_bf16(float a, float b) {
  bf16x2n p;
  p[0] = (__bf16)a;
  p[1] = (__bf16)b;
  return __builtin_bit_cast(uint32_t, p);
}

// 8 e4m3 values, scaled, to bf16
DEVINL u32x4v widen(uint64_t raw, float scale) {
  u32x4v r;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int b = (int)(uint32_t)(raw >> (32 * i));
    const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8(b, false);
    const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8(b, true);
    r[2 * i] = pack_bf16(lo[0] * scale, lo[1] * scale);
    r[2 * i + 1] = pack_bf16(hi[0] * scale, hi[1] * scale);
  }
  return r;
}

DEVINL void copy16_to_lds(const void* src, void* dst) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)src,
      (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

}  // namespace

// FIXED: the page size is 1 << bs_shift, of 16, 32 or 64 tokens, and a page of all
// heads has less than 2^32 values; otherwise the page size is bs_shift itself, a
// multiple of 8.
template <int D, bool KV_FP8, bool FIXED>
__global__ __launch_bounds__(PF_THREADS, D == 64 ? 3 : 2)
void prefill_attention_kernel(
    uint16_t* __restrict__ out,            // [T, Hq, D]
    float* __restrict__ tmp_acc,           // [T, Hq, splits, D] or null
    float* __restrict__ tmp_ml,            // [T, Hq, splits, 2]
    const uint16_t* __restrict__ q,        // [T, Hq, D], rows at q_stride
    const void* __restrict__ k_cache,      // [NB, Hk, BS, D]
    const void* __restrict__ v_cache,      // [NB, Hk, D, BS]
    const int* __restrict__ block_tables,  // [B, max_blocks]
    const int* __restrict__ seq_lens,      // [B] context with the portion
    const int* __restrict__ query_lens,    // [B] rows of the portion
    const int B, const int T, const int max_tiles, const int max_blocks,
    const int Hq, const int Hk, const int bs_shift, const int64_t q_stride,
    const float scale, const int window, const float softcap,
    const float* __restrict__ sinks, const float k_scale, const float v_scale) {
  constexpr int KCH = D / 8;                    // 16-byte chunks of a K row
  constexpr int KPER = PF_KT * KCH / PF_THREADS;  // chunks a thread stages
  constexpr int VPER = D * 8 / PF_THREADS;
  constexpr int KSTEPS = D / 16;
  constexpr int DT = D / 32;

  __shared__ __attribute__((aligned(16))) uint16_t K0[PF_KT * D];
  __shared__ __attribute__((aligned(16))) uint16_t V0[PF_KT * D];
  __shared__ __attribute__((aligned(16))) uint16_t K1[PF_KT * D];
  __shared__ __attribute__((aligned(16))) uint16_t V1[PF_KT * D];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  const int l31 = lane & 31;
  const int G = Hq / Hk;

  // Blocks are dealt round-robin to the 8 XCDs: with the key/value head as the
  // fastest index, the blocks that read one head's K and V share an XCD's L2
  // when 8 divides Hk. The last tiles of a causal portion see the most keys
  // and come first.
  const int hk = blockIdx.x % Hk;
  int tile = max_tiles - 1 - blockIdx.x / Hk;

  // which request: prefix sums over the portions, 64 at a time
  int req = -1, q0 = 0, QL = 0;
  {
    int tiles_before = 0, rows_before = 0;
    for (int b0 = 0; b0 < B; b0 += 64) {
      const int b = b0 + lane;
      const int ql = b < B ? max(query_lens[b], 0) : 0;
      const int nt = (ql * G + PF_ITEMS - 1) / PF_ITEMS;
      int tsum = nt, rsum = ql;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int t2 = __shfl_up(tsum, o, WAVE_SIZE);
        const int r2 = __shfl_up(rsum, o, WAVE_SIZE);
        if (lane >= o) {
          tsum += t2;
          rsum += r2;
        }
      }
      const int t_in = tile - tiles_before;
      const unsigned long long hit =
          __ballot(t_in >= tsum - nt && t_in < tsum);
      if (hit) {
        const int src = __ffsll(hit) - 1;
        req = b0 + src;
        QL = __shfl(ql, src, WAVE_SIZE);
        q0 = rows_before + __shfl(rsum, src, WAVE_SIZE) - QL;
        tile = t_in - (__shfl(tsum, src, WAVE_SIZE) -
                       __shfl(nt, src, WAVE_SIZE));
        break;
      }
      tiles_before += __shfl(tsum, 63, WAVE_SIZE);
      rows_before += __shfl(rsum, 63, WAVE_SIZE);
    }
  }
  if (req < 0) return;  // the grid is an upper bound
  req = __builtin_amdgcn_readfirstlane(req);
  QL = __builtin_amdgcn_readfirstlane(QL);
  q0 = __builtin_amdgcn_readfirstlane(q0);
  tile = __builtin_amdgcn_readfirstlane(tile);

  const int L = seq_lens[req];
  const int prefix = L - QL;
  const int items = QL * G;
  const int* btab = block_tables + (size_t)req * max_blocks;

  const int item = tile * PF_ITEMS + wid * 32 + l31;
  const int row = min(item, items - 1) / G;
  const int h = hk * G + min(item, items - 1) - row * G;
  const bool item_ok = item < items && q0 + row < T;
  const int qpos = prefix + row;
  // positions of the wave's first and last item, and of the workgroup's
  const int w0 = tile * PF_ITEMS + wid * 32;
  const bool wave_on = w0 < items;
  const int wpos_lo = prefix + min(w0, items - 1) / G;
  const int wpos_hi = prefix + min(w0 + 31, items - 1) / G;
  const int pos_lo = prefix + tile * PF_ITEMS / G;
  const int pos_hi =
      prefix + min(tile * PF_ITEMS + PF_ITEMS - 1, items - 1) / G;

  int kt_begin = 0;
  if (window > 0) kt_begin = max(0, pos_lo - window + 1) / PF_KT;
  int kt_end = (min(L, pos_hi + 1) + PF_KT - 1) / PF_KT;
  if (tmp_acc != nullptr) {
    const int per = (kt_end - kt_begin + gridDim.y - 1) / gridDim.y;
    kt_begin += blockIdx.y * per;
    kt_end = min(kt_end, kt_begin + per);
  }
  if (kt_begin >= kt_end) {  // no keys: nothing is looked up or copied
    if (half == 0 && item_ok) {
      const size_t at = (size_t)(q0 + row) * Hq + h;
      if (tmp_acc != nullptr) {
        float* ml = tmp_ml + (at * gridDim.y + blockIdx.y) * 2;
        ml[0] = kLowest;
        ml[1] = 0.f;
      } else {  // a portion longer than its context: 0 / 0, 0 beside a sink
        const uint32_t v = sinks != nullptr ? 0u : 0x7fc07fc0u;
        for (int d = 0; d < D; d += 4)
          *reinterpret_cast<uint2*>(out + at * D + d) = make_uint2(v, v);
      }
    }
    return;
  }

  // ---- Q as B operands: item l31, d = 16 s + 8 half + (0..7) -------------------
  bf16x8v qf[KSTEPS];
  {
    const uint16_t* qrow =
        q + (size_t)min(q0 + row, T - 1) * q_stride + h * D + half * 8;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      u32x4v v = {0, 0, 0, 0};
      if (item_ok) v = *reinterpret_cast<const u32x4v*>(qrow + s * 16);
      if (scale < 0.f) v ^= 0x80008000u;  // the sign goes with q
      qf[s] = __builtin_bit_cast(bf16x8v, v);
    }
  }
  // scores in units of log2: exp2(c * s - m); c > 0 also for a scale of 0, as
  // hidden scores are multiplied by it too
  const float c =
      softcap > 0.f ? 1.f : fmaxf(fabsf(scale) * kLog2e, 1e-20f);

  f32x16v o[DT] = {};
  float m = kLowest, l = 0.f;  // l: this half's tokens only

  // ---- tile addresses -----------------------------------------------------------
  // 16 chunks (256 bytes) make a turn over the banks: a K row of 128 values,
  // or two of 64; a V row has 64 tokens, so two as well
  auto k_swz = [](int r) { return D == 128 ? r & 15 : (r >> 1) & 7; };
  const int BS = FIXED ? 1 << bs_shift : bs_shift;
  const uint32_t page_elems = (uint32_t)Hk * BS * D;  // FIXED only
  // chunk i of a thread: its row of the tile and the chunk that belongs there
  auto k_row = [&](int i) { return ((wid * KPER + i) * 64 + lane) / KCH; };
  auto k_src = [&](int i) { return (lane % KCH) ^ k_swz(k_row(i)); };
  auto v_row = [&](int i) { return (wid * VPER + i) * 8 + (lane >> 3); };
  auto v_src = [&](int i) { return (lane & 7) ^ ((v_row(i) >> 1) & 7); };
  // FIXED: 16 K rows of a wave lie in one page, a V chunk column changes with
  // the parity of i only, and the place in a page is the same for every tile.
  // Page numbers are fetched a turn ahead of the copies that need them.
  // Tokens past the end are hidden later; their addresses stay inside a page
  // of the sequence.
  int koff[KPER], voff[VPER];
  if (FIXED) {
#pragma unroll
    for (int i = 0; i < KPER; ++i)
      koff[i] = (hk * BS + (k_row(i) & (BS - 1))) * D + k_src(i) * 8;
#pragma unroll
    for (int i = 0; i < VPER; ++i)
      voff[i] = (hk * D + v_row(i)) * BS + ((v_src(i) * 8) & (BS - 1));
  }
  int kpage = 0, vpage[2] = {0, 0};
  auto page_of_k = [&](int kt) {
    return FIXED ? btab[min(kt * PF_KT + wid * 16, L - 1) >> bs_shift] : 0;
  };
  auto pages = [&](int kt, int vt) {  // of K's tile kt and V's tile vt
    if (!FIXED) return;
    kpage = page_of_k(kt);
    vpage[0] = btab[min(vt * PF_KT + v_src(0) * 8, L - 1) >> bs_shift];
    vpage[1] = btab[min(vt * PF_KT + v_src(1) * 8, L - 1) >> bs_shift];
  };
  auto k_elem = [&](int kt, int i) -> size_t {
    if (FIXED) return (uint64_t)(uint32_t)kpage * page_elems + (uint32_t)koff[i];
    const int tok = min(kt * PF_KT + k_row(i), L - 1);
    return (size_t)btab[tok / BS] * Hk * BS * D + (hk * BS + tok % BS) * D +
           k_src(i) * 8;
  };
  auto v_elem = [&](int vt, int i) -> size_t {
    if (FIXED)
      return (uint64_t)(uint32_t)vpage[i & 1] * page_elems + (uint32_t)voff[i];
    // eight tokens of one page: BS is a multiple of 8
    const int tok = min(vt * PF_KT + v_src(i) * 8, (L - 1) & ~7);
    return (size_t)btab[tok / BS] * Hk * BS * D + (hk * D + v_row(i)) * BS +
           tok % BS;
  };
  auto copy_k = [&](int kt, uint16_t* Kl, int i) {
    copy16_to_lds((const uint16_t*)k_cache + k_elem(kt, i),
                  Kl + (wid * KPER + i) * 512);
  };
  auto copy_v = [&](int vt, uint16_t* Vl, int i) {
    copy16_to_lds((const uint16_t*)v_cache + v_elem(vt, i),
                  Vl + (wid * VPER + i) * 512);
  };
  auto issue_k = [&](int kt, uint16_t* Kl) {
#pragma unroll
    for (int i = 0; i < KPER; ++i) copy_k(kt, Kl, i);
  };
  auto issue_v = [&](int vt, uint16_t* Vl) {
#pragma unroll
    for (int i = 0; i < VPER; ++i) copy_v(vt, Vl, i);
  };
  uint64_t kraw[KV_FP8 ? KPER : 1], vraw[KV_FP8 ? VPER : 1];
  auto fetch_k = [&](int kt) {
#pragma unroll
    for (int i = 0; i < KPER; ++i)
      kraw[i] = *reinterpret_cast<const uint64_t*>((const uint8_t*)k_cache +
                                                   k_elem(kt, i));
  };
  auto fetch_v = [&](int vt) {
#pragma unroll
    for (int i = 0; i < VPER; ++i)
      vraw[i] = *reinterpret_cast<const uint64_t*>((const uint8_t*)v_cache +
                                                   v_elem(vt, i));
  };
  auto widen_k = [&](uint16_t* Kl) {
#pragma unroll
    for (int i = 0; i < KPER; ++i)
      *reinterpret_cast<u32x4v*>(Kl + ((wid * KPER + i) * 64 + lane) * 8) =
          widen(kraw[i], k_scale);
  };
  auto widen_v = [&](uint16_t* Vl) {
#pragma unroll
    for (int i = 0; i < VPER; ++i)
      *reinterpret_cast<u32x4v*>(Vl + ((wid * VPER + i) * 64 + lane) * 8) =
          widen(vraw[i], v_scale);
  };

  // operand rows: K row with bits 2 and 3 swapped (see the top), V row d
  const int krow = (l31 & 0x13) | ((l31 & 4) << 1) | ((l31 & 8) >> 1);
  auto k_frag = [&](const uint16_t* Kl, int ks, int t) {
    const int pos = (2 * ks + half) ^ k_swz(krow);
    return *reinterpret_cast<const bf16x8v*>(Kl + (t * 32 + krow) * D + pos * 8);
  };
  auto v_frag = [&](const uint16_t* Vl, int ks, int t) {
    const int d = t * 32 + l31;
    const int pos = (2 * ks + half) ^ ((d >> 1) & 7);
    return *reinterpret_cast<const bf16x8v*>(Vl + d * PF_KT + pos * 8);
  };

  float lsum = 0.f;
  float mx = kLowest;  // of the scores whose weights come next
  // weights of two tokens, part j of a B operand of 16
  auto weigh = [&](const f32x16v (&s)[2], int ks, int j) {
    const int r = (ks & 1) * 8 + 2 * j;
    const float a = __builtin_amdgcn_exp2f(fmaf(s[ks >> 1][r], c, -m));
    const float b = __builtin_amdgcn_exp2f(fmaf(s[ks >> 1][r + 1], c, -m));
    lsum += a;
    lsum += b;
    return pack_bf16(a, b);
  };
  auto larger = [&](float mx, const f32x16v& s) {
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
    return mx;
  };
  // rescaled when a maximum moved: its own weight is then 1, without rounding (only
  // when it moved by 2^8: 2% more error)
  auto raise = [&](float mx) {
    if (__any(mx > m)) {
      const float m2 = fmaxf(m, mx);
      const float f = __builtin_amdgcn_exp2f(m - m2);
      m = m2;
      l *= f;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] *= f;
    }
  };

  // ---- the tiles ------------------------------------------------------------------
  // The tiles that this wave's items see; the others are copied for the rest of the
  // workgroup.
  int on_begin = kt_begin, on_end = min(kt_end, (wpos_hi >> 6) + 1);
  if (window > 0) on_begin = max(on_begin, (wpos_lo - window + 1) >> 6);
  if (!wave_on) on_end = on_begin;

  auto hide = [&](int kbase, f32x16v (&s)[2]) {  // what the mask leaves out
    int last = qpos - kbase - 8 * half;  // the last token that is seen
    asm volatile("" : "+v"(last));  // not computed where no mask is applied
    const int first = window > 0 ? last - window : -1 << 30;  // and the one before all
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int tok = 32 * t + 16 * (r >> 3) + (r & 7);
        s[t][r] = tok <= last && tok > first ? s[t][r] : kHidden;
      }
  };

  // tiles of [inner, outer) are seen whole
  const int outer = (wpos_lo + 1) >> 6;
  const int inner = window > 0 ? ((wpos_hi - window) >> 6) + 1 : 0;

  // A turn takes the scores of tile kt and the weights and values of tile kt - 1.
  // One barrier a turn: behind it K of tile kt and V of tile kt - 1 are in LDS, and
  // every wave has left the buffers that the next ones go to.
  auto meet = [&](auto left) {  // copies of this thread that may be under way
    constexpr int n = decltype(left)::value;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070 | n);  // and lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  using none = std::integral_constant<int, 0>;
  f32x16v s0[2] = {}, s1[2];

  // Any turn: also the first and the last of this wave's tiles, a softcap, a mask.
  auto cut_turn = [&](int kt, const uint16_t* Kl, uint16_t* Kn, const uint16_t* Vl,
                      uint16_t* Vn) {
    const int kbase = kt * PF_KT;
    const bool more = kt < kt_end, first = kt == kt_begin;
    if (first) meet(std::integral_constant<int, KV_FP8 ? 0 : KPER + VPER>{});
    else meet(none{});
    if (more) {  // past the last tile K's copy is the last again
      if (first) {
      } else if (KV_FP8) {
        fetch_k(min(kt + 1, kt_end - 1));
        fetch_v(kt);
      } else {
        issue_k(min(kt + 1, kt_end - 1), Kn);
        issue_v(kt, Vn);
      }
      pages(min(kt + 2, kt_end - 1), kt + 1);
    }
    if (kt > on_begin && kt <= on_end) {
      raise(mx);
      const int n = L - kbase + PF_KT - 8 * half;  // tokens from this half's first
      const bool past = kbase > L;
#pragma unroll
      for (int ks = 0; ks < PF_KT / 16; ++ks) {
        u32x4v w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = weigh(s0, ks, j);
        bf16x8v a[DT];
#pragma unroll
        for (int t = 0; t < DT; ++t) a[t] = v_frag(Vl, ks, t);
        if (past) {  // a page's unused slots may hold anything
#pragma unroll
          for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int j = 0; j < 8; ++j)
              a[t][j] = 16 * ks + j < n ? a[t][j] : (short)0;
        }
#pragma unroll
        for (int t = 0; t < DT; ++t)
          o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              a[t], __builtin_bit_cast(bf16x8v, w), o[t], 0, 0, 0);
      }
      l += lsum;
      lsum = 0.f;
    }
    if (kt >= on_begin && kt < on_end) {
      s0[0] = s0[1] = f32x16v{};
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          s0[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k_frag(Kl, ks, t), qf[ks],
                                                          s0[t], 0, 0, 0);
      if (softcap > 0.f) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            s0[t][r] =
                softcap * tanhf(s0[t][r] * fabsf(scale) / softcap) * kLog2e;
      }
      if (kt < inner || kt >= outer) hide(kbase, s0);
      mx = max_halves(larger(larger(s0[0][0], s0[0]), s0[1])) * c;
    }
    if (KV_FP8 && more) {
      widen_k(Kn);
      if (!first) widen_v(Vn);
    }
  };

  // Tile kt seen whole, and tile kt - 1 one of this wave's. The order is the one that
  // is written here, a matrix instruction and what fits beside it at a time, operands
  // read AHEAD instructions early (2 to 8 measure the same); the compiler's own put
  // every read right before its use.
  auto whole_turn = [&](int kt, const uint16_t* Kl, uint16_t* Kn, const uint16_t* Vl,
                        uint16_t* Vn, f32x16v (&sn)[2], const f32x16v (&sp)[2]) {
    meet(none{});
    raise(mx);
    constexpr int S = 2 * KSTEPS, N = S + 4 * DT, AHEAD = 4;
    const int k_next = min(kt + 1, kt_end - 1), k_page = min(kt + 2, kt_end - 1);
    bf16x8v fr[AHEAD];
    u32x4v w[4];
    auto load = [&](int n) {
      fr[n % AHEAD] = n < S ? k_frag(Kl, n % KSTEPS, n / KSTEPS)
                            : v_frag(Vl, (n - S) / DT, (n - S) % DT);
    };
#pragma unroll
    for (int n = 0; n < AHEAD; ++n) load(n);
    if (KV_FP8) {
      fetch_k(k_next);
      fetch_v(kt);
      pages(k_page, kt + 1);
    }
#pragma unroll
    for (int n = 0; n < N; ++n) {
      __builtin_amdgcn_sched_barrier(0);
      if (n < S) {
        const int t = n / KSTEPS, ks = n % KSTEPS;
        sn[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            fr[n % AHEAD], qf[ks], ks ? sn[t] : f32x16v{}, 0, 0, 0);
      } else {
        const int t = (n - S) % DT, ks = (n - S) / DT;
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            fr[n % AHEAD], __builtin_bit_cast(bf16x8v, w[ks]), o[t], 0, 0, 0);
      }
      if (n + AHEAD < N) load(n + AHEAD);
      // 16 pairs of weights; each slice of four comes before its first product
#pragma unroll
      for (int u = 0; u < 16; ++u)
        if (u * (N - 4) / 16 == n) w[u / 4][u % 4] = weigh(sp, u / 4, u % 4);
      if (!KV_FP8) {
        if (n < KPER) copy_k(k_next, Kn, n);
        else if (n - KPER < VPER) copy_v(kt, Vn, n - KPER);
        else if (n == KPER + VPER) pages(k_page, kt + 1);
      }
      if (n == S) mx = larger(sn[0][0], sn[0]);
    }
    __builtin_amdgcn_sched_barrier(0);
    mx = max_halves(larger(mx, sn[1])) * c;
    l += lsum;
    lsum = 0.f;
    if (KV_FP8) {
      widen_k(Kn);
      widen_v(Vn);
    }
  };

  const int whole = max(on_begin + 1, inner);
  const int cut = softcap > 0.f ? 0 : min(on_end, outer);

  // The first turn's K, and behind it what that turn would ask for: the buffers are
  // free, and contexts of a few tiles are rows of such waits.
  pages(kt_begin, kt_begin);
  const int second = page_of_k(min(kt_begin + 1, kt_end - 1));
  if (KV_FP8) {
    fetch_k(kt_begin);
    fetch_v(kt_begin);
    kpage = second;
    widen_k(K0);
    widen_v(V0);
    fetch_k(min(kt_begin + 1, kt_end - 1));
  } else {
    issue_k(kt_begin, K0);
    asm volatile("" ::: "memory");
    kpage = second;
    issue_k(min(kt_begin + 1, kt_end - 1), K1);
    issue_v(kt_begin, V0);
  }
  for (int kt = kt_begin; kt <= kt_end; kt += 2) {
    if constexpr (D == 128) {
      for (; kt >= whole && kt + 1 < cut; kt += 2) {
        whole_turn(kt, K0, K1, V1, V0, s1, s0);
        whole_turn(kt + 1, K1, K0, V0, V1, s0, s1);
      }
    }
    cut_turn(kt, K0, K1, V1, V0);
    if (kt + 1 <= kt_end) cut_turn(kt + 1, K1, K0, V0, V1);
  }

  // ---- out: column = item, rows of O^T = d ---------------------------------------
  if (!item_ok) return;
  l = sum_halves(l);
  const size_t at = (size_t)(q0 + row) * Hq + h;
  if (tmp_acc != nullptr) {
    const size_t part = at * gridDim.y + blockIdx.y;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x4v v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = o[t][4 * i + r];
        *reinterpret_cast<f32x4v*>(tmp_acc + part * D + t * 32 + 8 * i +
                                   4 * half) = v;
      }
    if (half == 0) {
      tmp_ml[part * 2] = m * kLn2;
      tmp_ml[part * 2 + 1] = l;
    }
    return;
  }
  if (sinks != nullptr) l += __expf(sinks[h] - m * kLn2);
  const float inv = 1.f / l;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint2 v;
      v.x = pack_bf16(o[t][4 * i] * inv, o[t][4 * i + 1] * inv);
      v.y = pack_bf16(o[t][4 * i + 2] * inv, o[t][4 * i + 3] * inv);
      *reinterpret_cast<uint2*>(out + at * D + t * 32 + 8 * i + 4 * half) = v;
    }
}

// Upper bound of the tiles of B portions with T rows together.
extern "C" int prefill_attention_tiles(int T, int B, int Hq, int Hk) {
  return (int)(((long long)T * (Hq / Hk)) / PF_ITEMS) + B;
}

extern "C" void launch_prefill_attention(
    void* out, float* tmp_acc, float* tmp_ml, const void* q,
    const void* k_cache, const void* v_cache, const int* block_tables,
    const int* seq_lens, const int* query_lens, int T, int B, int Hq, int Hk,
    int D, int BS, int max_blocks, int64_t q_stride, float scale,
    int sliding_window, float softcap, const float* sinks, int splits,
    bool kv_fp8, float k_scale, float v_scale, hipStream_t stream,
    bool* launched) {
  *launched = false;
  const int max_tiles = prefill_attention_tiles(T, B, Hq, Hk);
  const bool fixed =
      (BS == 16 || BS == 32 || BS == 64) && (int64_t)Hk * BS * D < 1ll << 32;
  const int bs = fixed ? __builtin_ctz(BS) : BS;
  dim3 grid(max_tiles * Hk, splits, 1);
#define PF_LAUNCH(HD, FP8, P2)                                               \
  prefill_attention_kernel<HD, FP8, P2><<<grid, PF_THREADS, 0, stream>>>(    \
      (uint16_t*)out, tmp_acc, tmp_ml, (const uint16_t*)q, k_cache, v_cache, \
      block_tables, seq_lens, query_lens, B, T, max_tiles, max_blocks, Hq,   \
      Hk, bs, q_stride, scale, sliding_window, softcap, sinks, k_scale,      \
      v_scale);                                                              \
  *launched = true;
#define PF_LAUNCH2(HD, FP8)              \
  if (fixed) { PF_LAUNCH(HD, FP8, true) } \
  else { PF_LAUNCH(HD, FP8, false) }
  if (D == 128 && kv_fp8) { PF_LAUNCH2(128, true) }
  else if (D == 128) { PF_LAUNCH2(128, false) }
  else if (D == 64 && kv_fp8) { PF_LAUNCH2(64, true) }
  else if (D == 64) { PF_LAUNCH2(64, false) }
#undef PF_LAUNCH
#undef PF_LAUNCH2
}
