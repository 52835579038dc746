// Decode attention over listed tokens (MSA): each sequence (and key/value head)
// attends to the token positions of its list. The GQA query group rides the
// matrix cores:
//   S^T[64 tok x 16q] = K_tile . Q^T   A-frag: 8 consecutive d of one token
//   O^T[D x 16q]     += V^T . P        A-frag: 8 listed tokens of one d
// Q lives in registers; only P and the softmax reductions use LDS. K fragments
// are register double-buffered across tiles with NAMED buffers (a runtime-indexed
// buffer array goes to scratch). V is gathered per element, since listed tokens
// are not contiguous, at tile start so its latency hides under QK+softmax.
//
// One workgroup per (sequence, kv_head).

#include "common.h"

#define DM_THREADS 256

template <int HEAD_DIM, int BLOCK_SIZE>
__global__ __launch_bounds__(DM_THREADS) void msa_decode_kernel(
    uint16_t* __restrict__ out,        // [B, Hq, D]
    const uint16_t* __restrict__ q,    // [B, Hq, D] rows at q_stride
    const uint16_t* __restrict__ k_cache,  // [NB, Hk, BS, D]
    const uint16_t* __restrict__ v_cache,  // [NB, Hk, D, BS] (transposed)
    const int* __restrict__ block_tables,
    const int* __restrict__ seq_lens,
    const int max_blocks, const int Hk, const int G, const int64_t q_stride,
    const float scale,
    const int* __restrict__ token_positions,  // [B(,Hk), max_pos]
    const int max_positions, const int pos_heads) {
  constexpr int KT = 64;  // list entries a tile
  const int seq = blockIdx.y;
  const int hk = blockIdx.x;
  const int L = seq_lens[seq];
  const int* pos_row =
      token_positions +
      ((size_t)seq * pos_heads + (pos_heads > 1 ? hk : 0)) * max_positions;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = tid >> 6;
  const int l15 = lane & 15;
  const int l4 = lane >> 4;

  if (max_positions <= 0) return;

  __shared__ uint16_t Pl[16 * KT];  // row = q head, swz
  __shared__ float m_s[16], l_s[16], resc[16];
  __shared__ float wred[4][16];

  constexpr int KC = HEAD_DIM / 32;      // 16-B K/Q chunks per row
  constexpr int MT = HEAD_DIM / 16 / 4;  // PV M-tiles per wave
  constexpr int MS = KT / 64;            // token m-tiles per wave (QK)
  constexpr int SC = KT / 32;            // PV K-steps

  // ---- Q fragments in registers (head l15; zero-pad heads >= G) ---------------
  bf16x8v qfrag[KC];
  {
    const bool ok = l15 < G;
#pragma unroll
    for (int s = 0; s < KC; ++s) {
      int4 val = make_int4(0, 0, 0, 0);
      if (ok)
        val = *reinterpret_cast<const int4*>(
            q + (size_t)seq * q_stride + (hk * G + l15) * HEAD_DIM + s * 32 +
            l4 * 8);
      qfrag[s] = *reinterpret_cast<const bf16x8v*>(&val);
    }
  }
  if (tid < 16) {
    m_s[tid] = -3.0e4f;
    l_s[tid] = 0.f;
  }

  f32x4v acc_o[MT] = {};
  const int* btab = block_tables + (size_t)seq * max_blocks;
  const int kt_end = (max_positions + KT - 1) / KT;

  // list entry -> token (clamped for address safety — masked scores / zero p
  // neutralize the values)
  auto map_tok = [&](int j) -> int {
    const int gt = j < max_positions ? pos_row[j] : 0;
    return min(max(gt, 0), L - 1);
  };

  // K: wave wid owns token rows [wid*16*MS, +16*MS); lane l15 picks the row
  // within each 16-row m-tile, all KC d-chunks per row.
  int4 kregA[MS][KC], kregB[MS][KC];
  // V^T: lane covers d rows (wid*MT+mt)*16 + l15, token chunk s*32 + l4*8.
  int4 vreg[SC][MT];

  auto load_k = [&](int kt, int4 (&kreg)[MS][KC]) {
#pragma unroll
    for (int ms = 0; ms < MS; ++ms) {
      const int gtok = map_tok(kt * KT + (wid * MS + ms) * 16 + l15);
      const int blk = btab[gtok / BLOCK_SIZE];
      const size_t row =
          (((size_t)blk * Hk + hk) * BLOCK_SIZE + gtok % BLOCK_SIZE) * HEAD_DIM;
#pragma unroll
      for (int s = 0; s < KC; ++s)
        kreg[ms][s] =
            *reinterpret_cast<const int4*>(k_cache + row + s * 32 + l4 * 8);
    }
  };

  auto load_v = [&](int kt) {
#pragma unroll
    for (int s = 0; s < SC; ++s) {
      const int j0 = kt * KT + s * 32 + l4 * 8;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int drow = (wid * MT + mt) * 16 + l15;
        // listed tokens are scattered: per-element gather
        alignas(16) uint16_t e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int gt = map_tok(j0 + j);
          const int blk = btab[gt / BLOCK_SIZE];
          e[j] = v_cache[(((size_t)blk * Hk + hk) * HEAD_DIM + drow) * BLOCK_SIZE +
                         gt % BLOCK_SIZE];
        }
        vreg[s][mt] = *reinterpret_cast<const int4*>(e);
      }
    }
  };

  auto tile_math = [&](int kt, const int4 (&kreg)[MS][KC]) {
    const int kbase = kt * KT;

    // ---- S^T = K . Q^T (wave w: token rows [w*16*MS, +16*MS)) -------------------
    f32x4v acc_s[MS] = {};
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ms = 0; ms < MS; ++ms)
#pragma unroll
      for (int s = 0; s < KC; ++s) {
        const bf16x8v afrag = *reinterpret_cast<const bf16x8v*>(&kreg[ms][s]);
        acc_s[ms] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            afrag, qfrag[s], acc_s[ms], 0, 0, 0);
      }
    __builtin_amdgcn_s_setprio(0);

    // ---- mask + per-column max --------------------------------------------------
    float mx = -3.0e4f;
#pragma unroll
    for (int ms = 0; ms < MS; ++ms)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = kbase + (wid * MS + ms) * 16 + l4 * 4 + r;
        float s = acc_s[ms][r] * scale;
        bool visible = j < max_positions && l15 < G;
        if (visible) {
          const int gt = pos_row[j];
          visible = gt >= 0 && gt < L;
        }
        s = visible ? s : -3.0e4f;
        acc_s[ms][r] = s;
        mx = fmaxf(mx, s);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE_SIZE));
    mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE_SIZE));
    if (lane < 16) wred[wid][lane] = mx;
    __syncthreads();
    if (tid < 16) {
      const float m_chunk = fmaxf(fmaxf(wred[0][tid], wred[1][tid]),
                                  fmaxf(wred[2][tid], wred[3][tid]));
      const float m_new = fmaxf(m_s[tid], m_chunk);
      resc[tid] = __expf(m_s[tid] - m_new);
      m_s[tid] = m_new;
    }
    __syncthreads();

    // ---- p = exp(s - m) -> Pl; column sums ---------------------------------------
    float sm = 0.f;
    {
      const float m = m_s[l15];
#pragma unroll
      for (int ms = 0; ms < MS; ++ms)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = __expf(acc_s[ms][r] - m);
          sm += p;
          const int kk = (wid * MS + ms) * 16 + l4 * 4 + r;
          const int pb = swz(l15 * KT * 2 + kk * 2, l15);
          *reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(Pl) + pb) =
              f32_to_bf16_bits(p);
        }
      sm += __shfl_xor(sm, 16, WAVE_SIZE);
      sm += __shfl_xor(sm, 32, WAVE_SIZE);
    }
    if (lane < 16) wred[wid][lane] = sm;
    __syncthreads();  // Pl + wred writes from every wave before l_s / PV
    if (tid < 16)
      l_s[tid] = l_s[tid] * resc[tid] + wred[0][tid] + wred[1][tid] +
                 wred[2][tid] + wred[3][tid];

    // ---- O^T += V^T . P ----------------------------------------------------------
    {
      const float r = resc[l15];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) acc_o[mt][rr] *= r;
    }
    // barrier: l_s's wred read + everyone's resc read must complete before
    // the next tile's wred/resc writes (threads race ahead through PV)
    __syncthreads();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < SC; ++s) {
      const int pb = swz(l15 * KT * 2 + s * 64 + l4 * 16, l15);
      const bf16x8v bfrag = *reinterpret_cast<const bf16x8v*>(
          reinterpret_cast<const char*>(Pl) + pb);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const bf16x8v afrag = *reinterpret_cast<const bf16x8v*>(&vreg[s][mt]);
        acc_o[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afrag, bfrag,
                                                            acc_o[mt], 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
    // no trailing barrier: the next tile's two reduction barriers precede any
    // Pl/resc rewrite, so this tile's PV reads are already protected
  };

  load_k(0, kregA);
  for (int kt = 0; kt < kt_end; ++kt) {
    // V for THIS tile issues first (its latency hides under QK+softmax);
    // next tile's K prefetches into the other named buffer.
    load_v(kt);
    if ((kt & 1) == 0) {
      if (kt + 1 < kt_end) load_k(kt + 1, kregB);
      tile_math(kt, kregA);
    } else {
      if (kt + 1 < kt_end) load_k(kt + 1, kregA);
      tile_math(kt, kregB);
    }
  }

  // ---- write out (O^T acc: col=q head, row=d) -----------------------------------
  const int g = l15;
  if (g < G) {
    const size_t hq = (size_t)hk * G + g;
    const float inv = 1.f / l_s[g];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int d0 = (wid * MT + mt) * 16 + l4 * 4;
      uint16_t vals[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) vals[r] = f32_to_bf16_bits(acc_o[mt][r] * inv);
      *reinterpret_cast<uint2*>(out + hq * HEAD_DIM +
                                (size_t)seq * Hk * G * HEAD_DIM + d0) =
          *reinterpret_cast<const uint2*>(vals);
    }
  }
}

extern "C" void launch_msa_paged_attention_decode(
    void* out, const void* q, const void* k_cache, const void* v_cache,
    const int* block_tables, const int* seq_lens, const int* token_positions,
    int max_positions, int pos_heads, int B, int Hq, int Hk, int D, int BS,
    int max_blocks, int64_t q_stride, float scale, hipStream_t stream,
    bool* launched) {
  const int G = Hq / Hk;
  *launched = false;
  if (G > 16) return;
  dim3 grid(Hk, B, 1);
#define MSA_LAUNCH(HD, BSZ)                                                    \
  msa_decode_kernel<HD, BSZ><<<grid, DM_THREADS, 0, stream>>>(                 \
      (uint16_t*)out, (const uint16_t*)q, (const uint16_t*)k_cache,            \
      (const uint16_t*)v_cache, block_tables, seq_lens, max_blocks, Hk, G,     \
      q_stride, scale, token_positions, max_positions, pos_heads);             \
  *launched = true;
  if (D == 128 && BS == 32) { MSA_LAUNCH(128, 32) }
  else if (D == 128 && BS == 16) { MSA_LAUNCH(128, 16) }
  else if (D == 128 && BS == 64) { MSA_LAUNCH(128, 64) }
  else if (D == 64 && BS == 32) { MSA_LAUNCH(64, 32) }
  else if (D == 64 && BS == 16) { MSA_LAUNCH(64, 16) }
  else if (D == 64 && BS == 64) { MSA_LAUNCH(64, 64) }
#undef MSA_LAUNCH
}
