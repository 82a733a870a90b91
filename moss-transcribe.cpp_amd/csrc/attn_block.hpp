// attn_block.hpp - attention of a block of query rows on f32 MFMA, for the causal
// prefill (head_dim 128, a KV cache in f32 or f16) and the audio encoder (head_dim
// 64, no mask). Results follow the canonical order (device_common.hpp): chunks of
// 64 keys, each score an fma chain over head_dim, p = exp(w - m_c), l_c the
// butterfly sum, O_c an fma chain over the chunk's keys, chunks merged in order
// with f_c = exp(m_c - M), M the row's maximum over all keys.
//
// What bounds it: v_mfma_f32_16x16x4f32 takes 33 cycles per SIMD and does not run
// beside f32 vector instructions (measured: 33 cycles plus 4-5 per fma), so the
// time is the sum of the MFMAs and of every vector instruction. Hence
//   * M comes from an estimate instead of a first exact pass over all scores: f16
//     MFMA (18 cycles for eight times the products) finds each row's best keys,
//     only those scores are computed exactly, and the exact pass checks that no
//     score exceeded M; if one did, the pass is repeated with the true maximum.
//   * each K and V operand register feeds two query tiles (the two q heads of a kv
//     head, or two row tiles of an encoder head);
//   * V needs no transpose: output row i of P.V tile dt is element NDT * i + dt, so a
//     lane's operands for all dt are contiguous in memory and load straight into
//     registers. K goes through a wave-private LDS tile (16 keys), no barrier.
// A workgroup takes 2 query tiles of 16; its four waves take chunks c = wave mod 4.
// Every chunk's (l_c, O_c) is computed independently; the running (L, O) travels
// from wave to wave through LDS in chunk order (the merge is 1 / 16 of the work).
// Two workgroups per CU, two waves per SIMD (head_dim 64: three; the encoder's 24 layers
// 7.29 -> 7.19 ms). With an f32 cache the 256 registers do not hold everything: 13 or 14
// are spilled, of which a chunk reloads four; the encoder's form spills 10 of its 168, the
// f16-cache forms none.
// Measured (kernel trace) against two exact passes with K and V^T staged by the whole
// workgroup: 1,600 rows, f32 cache 289 -> 203 us per layer (the MFMAs alone: 69 us; the
// rest is the estimates' reads of K at the start, vector work and the uneven causal
// blocks); 2,048 rows after 14,336, f16 cache 3.80 -> 2.73 ms, 2.59 to 3.11 (1.64 ms); the
// encoder's 1,500 rows x 16 heads 202 -> 153 us (60 us).
//
// What a repeat costs: the workgroup's exact pass once more. On noise, at most 0.3 % of the
// workgroups repeat; on constant, half constant and nearly constant prompts and mel chunks
// 2.6 % with an f32 cache (whole prefills up to 7 % longer) and 0.1 % with an f16 one.
// Where a head's keys score alike to within f16's resolution (rows equal to 3e-6 and every
// rotation but the slowest taken out of the keys), 25 to 81 % repeat with an f32 cache:
// 1,600 rows, 8 layers 7.4 -> 8.4 ms a prompt (two exact passes: 10.4), 8,000 rows, 4
// layers 24.9 -> 34.8 (35.0), but 16,384 rows, 4 layers 59.5 -> 98.8 (82.8), the one kind of
// input found on which two exact passes are faster. Giving a pass up at its first score
// above M (maxima only from there on) made that 93.0 and 1,600 rows no faster, and the
// registers it takes cost ordinary prompts of 16,384 rows 1.5 to 2.5 %.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "device_common.hpp"

namespace mtg {
namespace dev {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));

struct AttnBlockArgs {
  const float* q;       // [row][q_stride]
  const uint8_t* k;     // kv head h at + h * head_bytes, key i at + i * key_bytes
  const uint8_t* v;
  size_t head_bytes;
  int key_bytes;
  int q_stride, out_stride;  // floats
  int group;            // q heads per kv head (causal)
  int past, S, kvlen;   // rows 0 .. S - 1 at positions past + row; kvlen keys
  float* out;           // f32 rows [row][out_stride], or
  int8_t* ocodes;       // q8_0 codes and scales of rows of q_stride (q8_rows_code, q8_rows_scale)
  float* oscales;
};

constexpr int kAbWaves = 4;
constexpr float kAbNone = -3.0e38f;  // below every estimate

template <int HD>
struct AbLds {
  static constexpr int NDT = HD / 16;
  static constexpr int ktile = 16 * HD;                         // floats per wave
  static constexpr int box = kAbWaves * ktile;                  // mailbox: O of 2 tiles, then L
  static constexpr int lrow = box + 2 * NDT * 64 * 4;           // [2][64]
  static constexpr int top = lrow + 128;                        // [wave][32 rows] maxima
  static constexpr int seq = top + kAbWaves * 32;
  static constexpr size_t bytes = (size_t)(seq + 4) * 4;
};

// canonical exp of a non-positive (or NaN) argument: dev_expf without its upper range
__device__ __forceinline__ float ab_exp_neg(float x) {
  const float n = rintf(__fmul_rn(x, 1.44269504f));
  float r = fmaf(n, -0.693145752f, x);
  r = fmaf(n, -1.42860677e-06f, r);
  float p = 1.98412698e-4f;
  p = fmaf(p, r, 1.38888889e-3f);
  p = fmaf(p, r, 8.33333333e-3f);
  p = fmaf(p, r, 4.16666667e-2f);
  p = fmaf(p, r, 1.66666667e-1f);
  p = fmaf(p, r, 0.5f);
  p = fmaf(p, r, 1.0f);
  p = fmaf(p, r, 1.0f);
  const float e = ldexpf(p, (int)fmaxf(n, -200.0f));
  return x < -87.0f ? 0.0f : e;
}

template <int KVH>
__device__ __forceinline__ void ab_halves(const v4i h, float (&f)[8]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f[2 * e] = half_bits_to_float((uint16_t)((uint32_t)h[e] & 0xffffu));
    f[2 * e + 1] = half_bits_to_float((uint16_t)((uint32_t)h[e] >> 16));
  }
}

// Eight elements of a row as an f16 MFMA operand (estimates only): lane group g takes
// elements 8 g .. 8 g + 7 of every 32 from f16 rows and 4 g .. 4 g + 3 of every 16
// from f32 rows, so that a load covers 64 contiguous bytes per row.
template <int KVH>
struct AbPiece {
  v4i r[KVH ? 1 : 2];
  __device__ __forceinline__ void load(const uint8_t* p) {
    r[0] = *(const v4i*)p;
    if constexpr (!KVH) r[1] = *(const v4i*)(p + 64);
  }
  __device__ __forceinline__ v8h get() const {
    if constexpr (KVH) {
      return __builtin_bit_cast(v8h, r[0]);
    } else {
      v8h o;
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = (_Float16)__int_as_float(r[i / 4][i % 4]);
      return o;
    }
  }
};

// CAUSAL: tiles are q heads 2 blockIdx.x + u of one kv head, rows r0 .. r0 + 15 at
// positions past + row. Else: rows r0 + 16 u .. of head blockIdx.x, every key.
// OUTQ: q8_0 codes and scales (HD == 128), else f32 rows.
template <int HD, int KVH, bool CAUSAL, bool OUTQ>
__global__ void __launch_bounds__(256, HD == 64 ? 3 : 2) k_attn_block(const AttnBlockArgs A) {
  using Lds = AbLds<HD>;
  constexpr int NDT = HD / 16, NS = HD / 4, ES = KVH ? 2 : 4;
  extern __shared__ float ab_lds[];
  const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int by = CAUSAL ? (int)(gridDim.y - 1 - blockIdx.y) : (int)blockIdx.y;  // the longest blocks first
  const int r0 = by * (CAUSAL ? 16 : 32);
  const int kvlen = A.kvlen, last_key = kvlen - 1;
  const int kvh = CAUSAL ? 2 * (int)blockIdx.x / A.group : (int)blockIdx.x;
  const uint8_t* kh = A.k + (size_t)kvh * A.head_bytes;
  const uint8_t* vh = A.v + (size_t)kvh * A.head_bytes;
  const int nch = (CAUSAL ? min(A.past + r0 + 15, last_key) : last_key) / kChunk + 1;
  const int full_to = CAUSAL ? A.past + r0 : last_key;  // chunks that end at or before this key need no mask
  const float scale = __fdiv_rn(1.0f, dev_sqrtf((float)HD));
  int row[2], qoff[2], pos[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    row[u] = CAUSAL ? r0 + j : r0 + 16 * u + j;
    qoff[u] = (CAUSAL ? 2 * (int)blockIdx.x + u : (int)blockIdx.x) * HD;
    pos[u] = CAUSAL ? A.past + row[u] : last_key;
  }

  // A 16-row tile in LDS: 4-element piece y of row i at y * 64 + (i ^ 2 (y & 7)) * 4
  // floats: writes (a row's pieces from neighbouring lanes) and reads (one piece or
  // element of 16 rows) both spread over all banks
  const int wkey = lane >> 2, wq = lane & 3;
  float* const sq = ab_lds + Lds::box;  // the two q tiles, until the mailbox is needed
  {
    const int u = wave & 1, qrow = CAUSAL ? r0 + wkey : r0 + 16 * u + wkey;
    const float* src = A.q + (size_t)min(qrow, A.S - 1) * A.q_stride +
                       (CAUSAL ? 2 * (int)blockIdx.x + u : (int)blockIdx.x) * HD + 4 * wq;
    v4f t[NS / 8];
#pragma unroll
    for (int x = 0; x < NS / 8; ++x) t[x] = *(const v4f*)(src + 16 * (2 * x + (wave >> 1)));
#pragma unroll
    for (int x = 0; x < NS / 8; ++x) {
      const int y = 4 * (2 * x + (wave >> 1)) + wq;
      *(v4f*)(sq + u * 16 * HD + y * 64 + (wkey ^ (2 * (y & 7))) * 4) = qrow < A.S ? t[x] : v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  // K tiles go through this wave's LDS tile in the same layout
  float* const sk = ab_lds + wave * Lds::ktile;
  constexpr int NKL = HD * ES / 64;  // 16-byte loads per lane and tile
  v4i kreg[NKL];
  auto k_load_rows = [&](const uint8_t* lane_row, v4i (&kr)[NKL]) {
#pragma unroll
    for (int x = 0; x < NKL; ++x) kr[x] = *(const v4i*)(lane_row + 16 * wq + 64 * x);
  };
  auto k_load = [&](int key) {  // keys key .., rows past the last key read the last one
    const int key0 = min(key, last_key);
    const uint8_t* base = kh + (size_t)key0 * A.key_bytes;
    k_load_rows(base + (uint32_t)(min(wkey, last_key - key0) * A.key_bytes), kreg);
  };
  auto k_store = [&](const v4i (&kr)[NKL]) {
#pragma unroll
    for (int x = 0; x < NKL; ++x) {
      if constexpr (KVH) {
        float f[8];
        ab_halves<KVH>(kr[x], f);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int y = 8 * x + 2 * wq + h;
          *(v4f*)(sk + y * 64 + (wkey ^ (2 * (2 * wq + h))) * 4) = v4f{f[4 * h], f[4 * h + 1], f[4 * h + 2], f[4 * h + 3]};
        }
      } else {
        const int y = 4 * x + wq;
        *(v4i*)(sk + y * 64 + (wkey ^ (2 * (4 * (x & 1) + wq))) * 4) = kr[x];
      }
    }
  };
  float qb[2][NS];

  const bool one_round = nch <= kAbWaves;  // every wave has one chunk at most: the exact pass shares its maxima

  // ---- the rows' maxima: estimates of every score, the exact scores of the best
  float* const s_top = ab_lds + Lds::top;
  {
    constexpr int TP = KVH ? 4 : 2, NX = HD / 32;  // key tiles per step, 32-element pieces per row
    v8h qh[2][NX];
    float b1[2] = {kAbNone, kAbNone}, b2[2] = {kAbNone, kAbNone};
    int i1[2] = {0, 0}, i2[2] = {0, 0};
    const int steps = one_round ? 0 : ((nch - wave + kAbWaves - 1) / kAbWaves) * (4 / TP);  // of this wave's chunks
    auto step_key = [&](int n) { return ((n / (4 / TP)) * kAbWaves + wave) * kChunk + (n % (4 / TP)) * 16 * TP; };
    AbPiece<KVH> nx[2][TP][NX];  // two steps in flight
    auto fetch = [&](int n, AbPiece<KVH> (&p)[TP][NX]) {
      const int key0 = step_key(n);
#pragma unroll
      for (int t = 0; t < TP; ++t) {
        const uint8_t* kr = kh + (size_t)min(key0 + 16 * t + j, last_key) * A.key_bytes + 16 * g;
#pragma unroll
        for (int x = 0; x < NX; ++x) p[t][x].load(kr + 32 * ES * x);
      }
    };
    auto step = [&](int n, AbPiece<KVH> (&p)[TP][NX]) {
      const int key0 = step_key(n);
      v4f e[2][TP];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int t = 0; t < TP; ++t) e[u][t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int x = 0; x < NX; ++x)
#pragma unroll
        for (int t = 0; t < TP; ++t) {
          const v8h a = p[t][x].get();
#pragma unroll
          for (int u = 0; u < 2; ++u) e[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qh[u][x], e[u][t], 0, 0, 0);
        }
      fetch(n + 2, p);  // past the last step: the last key's row
      __builtin_amdgcn_sched_barrier(0);
      const bool full = key0 + 16 * TP - 1 <= full_to;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float best = kAbNone;
#pragma unroll
        for (int t = 0; t < TP; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            // the key's place in the step replaces the lowest mantissa bits
            float c = __uint_as_float((__float_as_uint(e[u][t][r]) & ~15u) | (uint32_t)(4 * t + r));
            if (!full && key0 + 16 * t + 4 * g + r > pos[u]) c = kAbNone;
            best = fmaxf(best, c);
          }
        const bool first = best > b1[u], second = best > b2[u];
        i2[u] = first ? i1[u] : (second ? n : i2[u]);
        b2[u] = first ? b1[u] : (second ? best : b2[u]);
        i1[u] = first ? n : i1[u];
        b1[u] = first ? best : b1[u];
      }
    };
    if (steps > 0) {
      fetch(0, nx[0]);
      fetch(1, nx[1]);
    }
    __syncthreads();  // the q tiles are staged
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int x = 0; x < NX; ++x) {
        AbPiece<0> p;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int y = KVH ? 8 * x + 2 * g + h : 8 * x + 4 * h + g;
          p.r[h] = *(const v4i*)(sq + u * 16 * HD + y * 64 + (j ^ (2 * (y & 7))) * 4);
        }
        qh[u][x] = p.get();
      }
    for (int n = 0; n < steps; n += 2) {
      step(n, nx[0]);
      if (n + 1 < steps) step(n + 1, nx[1]);
    }
    // B operands of the exact scores: q[row][4 s + g] (f16-rounded for an f16 cache)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const float v = sq[u * 16 * HD + s * 64 + (j ^ (2 * (s & 7))) * 4 + g];
        qb[u][s] = KVH ? f16_round(v) : v;
      }
    // The wave's best key of every row (the best two of an f32 cache, whose estimates
    // round the operands): key j of a gathered tile is row j's, so its exact scores
    // are the diagonal of one tile's MFMA chain, lane (g, j) = (j / 4, j), register j % 4.
    constexpr int RANKS = KVH ? 1 : 2;
    if (!one_round) {
      float m[2] = {-INFINITY, -INFINITY};
      int ckey[RANKS][2];
      v4i creg[RANKS][2][NKL];
#pragma unroll
      for (int rank = 0; rank < RANKS; ++rank)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          float b = fmaxf(b1[u], lane_xor_f<16>(b1[u]));
          b = fmaxf(b, lane_xor_f<32>(b));
          const bool mine = b1[u] == b && b > kAbNone;
          const int id = (int)(__float_as_uint(b) & 15u);
          int key = mine ? step_key(i1[u]) + 16 * (id >> 2) + 4 * g + (id & 3) : -1;
          key = max(key, (int)lane_xor<16>((uint32_t)key));
          ckey[rank][u] = max(key, (int)lane_xor<32>((uint32_t)key));  // row j's key in every lane of column j
          if (mine) {  // the winner's next best takes its place
            b1[u] = b2[u];
            i1[u] = i2[u];
          }
          k_load_rows(kh + (size_t)max(__shfl(ckey[rank][u], wkey), 0) * A.key_bytes, creg[rank][u]);
        }
#pragma unroll
      for (int rank = 0; rank < RANKS; ++rank)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          k_store(creg[rank][u]);
          v4f d = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int s = 0; s < NS; ++s)
            d = __builtin_amdgcn_mfma_f32_16x16x4f32(sk[s * 64 + (j ^ (2 * (s & 7))) * 4 + g], qb[u][s], d, 0, 0, 0);
          const float e = (j & 2) ? ((j & 1) ? d[3] : d[2]) : ((j & 1) ? d[1] : d[0]);
          if (ckey[rank][u] >= 0) m[u] = fmaxf(m[u], __fmul_rn(e, scale));
        }
      if (g == j >> 2) {
        s_top[wave * 32 + j] = m[0];
        s_top[wave * 32 + 16 + j] = m[1];
      }
    }
    if (tid == 0) *(volatile int*)(ab_lds + Lds::seq) = 0;
    if (wave < nch) k_load(wave * kChunk);
    __syncthreads();
  }
  float M[2];
  auto row_maxima = [&]() {  // over the waves that have a chunk
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      M[u] = s_top[16 * u + j];
      for (int i = 1; i < min(nch, kAbWaves); ++i) M[u] = fmaxf(M[u], s_top[i * 32 + 16 * u + j]);
    }
  };
  if (!one_round) row_maxima();

  // ---- the exact pass
  // A row j of a key tile is key 4 (j % 4) + j / 4, so output register r of lane (g, j)
  // is key 4 r + g of the tile: the B operand of P.V step m = 4 t + r
  const int akey = 4 * (j & 3) + (j >> 2);
  const float* ka[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) ka[i] = sk + i * 64 + (akey ^ (2 * i)) * 4 + g;
  // V operands of step m, key 4 m + g: output row i of tile dt is element 8 i + dt (f16
  // rows) or 64 (dt / 4) + 4 i + dt % 4 (f32 rows), whole 16-byte pieces of a row
  constexpr int NVL = NDT * ES / 16;  // 16-byte loads per lane and step
  constexpr int VAHEAD = 4;
  v4i vreg[16][NVL];
  auto v_load = [&](int key0, int m) {
    const uint8_t* base = vh + (size_t)key0 * A.key_bytes;
    const uint32_t off = (uint32_t)(min(4 * m + g, last_key - key0) * A.key_bytes + 16 * j);
#pragma unroll
    for (int x = 0; x < NVL; ++x) vreg[m][x] = *(const v4i*)(base + off + 256 * x);
  };
  volatile int* const seq = (volatile int*)(ab_lds + Lds::seq);
  v4f* const box = (v4f*)(ab_lds + Lds::box);
  float* const lbox = ab_lds + Lds::lrow;

  for (int attempt = 0; attempt < 2; ++attempt) {
    float top[2] = {-INFINITY, -INFINITY};
    for (int c = wave; c < nch; c += kAbWaves) {
      const int key0 = c * kChunk;
      const bool full = key0 + kChunk - 1 <= full_to;
      v4f w[2][4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        k_store(kreg);
        __builtin_amdgcn_sched_barrier(0);
        if (t < 3) k_load(key0 + 16 * (t + 1));
        __builtin_amdgcn_sched_barrier(0);
        w[0][t] = w[1][t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int x = 0; x < NS / 8; x += 2) {
          float a[2][8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            a[0][i] = ka[i][x * 512];
            a[1][i] = ka[i][(x + 1) * 512];
          }
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
              for (int u = 0; u < 2; ++u)
                w[u][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[h][i], qb[u][8 * (x + h) + i], w[u][t], 0, 0, 0);
        }
      }
#pragma unroll
      for (int m = 0; m < VAHEAD; ++m) v_load(key0, m);
      __builtin_amdgcn_sched_barrier(0);
      // chunk softmax
      float mc[2], lc[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) w[u][t][r] = __fmul_rn(w[u][t][r], scale);
        if (!full) {
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (key0 + 16 * t + 4 * r + g > pos[u]) w[u][t][r] = -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) mx = fmaxf(mx, w[u][t][r]);
        mx = pair_max_f<32>(mx);
        mc[u] = pair_max_f<16>(mx);
        top[u] = fmaxf(top[u], mc[u]);
        // a row without a key in the chunk: every p is 0 (only in chunks with a mask, or of NaN)
        const float base = mc[u] == -INFINITY ? 0.0f : mc[u];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float pv = ab_exp_neg(__fsub_rn(w[u][t][r], base));
            w[u][t][r] = KVH ? f16_round(pv) : pv;
          }
        if (CAUSAL && __any(mc[u] == -INFINITY))
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) w[u][t][r] = mc[u] == -INFINITY ? 0.0f : w[u][t][r];
        // l_c: key levels 32, 16 (t), 8, 4 (r) in the lane, 2, 1 (g) across lanes
        float y[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          y[r] = __fadd_rn(__fadd_rn(w[u][0][r], w[u][2][r]), __fadd_rn(w[u][1][r], w[u][3][r]));
        lc[u] = pair_add_f<32>(__fadd_rn(__fadd_rn(y[0], y[2]), __fadd_rn(y[1], y[3])));
        lc[u] = pair_add_f<16>(lc[u]);
      }
      // P.V
      v4f oc[2][NDT];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) oc[u][dt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      const bool tail = key0 + kChunk - 1 > last_key;  // rows past the last key count as zeros
      float av[2][NDT];
      auto v_operands = [&](int m, int b) {
        if (tail && key0 + 4 * m + g > last_key)
#pragma unroll
          for (int x = 0; x < NVL; ++x) vreg[m][x] = v4i{0, 0, 0, 0};
        if constexpr (KVH) {
          static_assert(!KVH || NDT == 8, "f16 keys: head_dim 128");
          ab_halves<KVH>(vreg[m][0], *(float(*)[8])av[b]);
        } else {
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) av[b][dt] = __int_as_float(vreg[m][dt / 4][dt % 4]);
        }
      };
      v_operands(0, 0);
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        if (m + VAHEAD < 16) v_load(key0, m + VAHEAD);
        if (m == 16 - VAHEAD) k_load(key0 + kAbWaves * kChunk);  // the next chunk's first tile
        __builtin_amdgcn_sched_barrier(0);
        if (m < 15) v_operands(m + 1, (m + 1) & 1);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
          for (int u = 0; u < 2; ++u)
            oc[u][dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[m & 1][dt], w[u][m >> 2][m & 3], oc[u][dt], 0, 0, 0);
      }
      if (one_round) {
        if (g == 0) {
          s_top[wave * 32 + j] = mc[0];
          s_top[wave * 32 + 16 + j] = mc[1];
        }
        __syncthreads();
        row_maxima();
      }
      // merge: wait for chunk c - 1, then pass (L, O) on. Chunk c - 1 belongs to another
      // wave of this workgroup that waits only on earlier chunks, so every wait ends.
      float f[2];
#pragma unroll
      for (int u = 0; u < 2; ++u)
        f[u] = mc[u] == -INFINITY ? 0.0f : dev_expf(__fsub_rn(mc[u], M[u]));
      if (c > 0) {
        while (*seq != c) __builtin_amdgcn_s_sleep(1);
        asm volatile("" ::: "memory");
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const float L = lbox[u * 64 + lane];
          lbox[u * 64 + lane] = fmaf(lc[u], f[u], L);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            v4f O = box[(u * NDT + dt) * 64 + lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) O[r] = fmaf(oc[u][dt][r], f[u], O[r]);
            box[(u * NDT + dt) * 64 + lane] = O;
          }
        }
      } else {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          lbox[u * 64 + lane] = fmaf(lc[u], f[u], 0.0f);
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) {
            v4f O;
#pragma unroll
            for (int r = 0; r < 4; ++r) O[r] = fmaf(oc[u][dt][r], f[u], 0.0f);
            box[(u * NDT + dt) * 64 + lane] = O;
          }
        }
      }
      // the LDS serves a wave's accesses in order: (L, O) are stored before the count
      asm volatile("" ::: "memory");
      if (lane == 0) *seq = c + 1;
    }
    if (one_round) {
      if (wave >= nch) __syncthreads();  // the barrier of the waves with a chunk
      __syncthreads();
      break;
    }
    // the largest score of every row, against the maximum the merge used
    if (g == 0) {
      s_top[wave * 32 + j] = top[0];
      s_top[wave * 32 + 16 + j] = top[1];
    }
    __syncthreads();
    const float used[2] = {M[0], M[1]};
    row_maxima();
    const bool off = (row[0] < A.S && M[0] != used[0]) || (row[1] < A.S && M[1] != used[1]);
    if (!__syncthreads_or(off)) break;
    if (tid == 0) *seq = 0;
    k_load(wave * kChunk);
    __syncthreads();
  }

  // O[u][dt][r] of lane (g, j): output row i = 4 g + r of row[u] (the element: v_load)
  const int u = wave & 1, orow = u ? row[1] : row[0], ooff = u ? qoff[1] : qoff[0];
  const float L = lbox[u * 64 + lane];
  if constexpr (OUTQ) {
    static_assert(!OUTQ || HD == 128, "q8_0 blocks of a 128-element head");
    if (wave >= 2) return;
    // two runs of 16 elements in order: f16 rows 32 g .. and 32 g + 16 .., one q8_0 block;
    // f32 rows 16 g .. and 64 + 16 g .., halves of two blocks shared with lane g ^ 1
    float o[2][16];
    uint32_t top[2] = {0, 0};
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      const v4f O = box[(u * NDT + dt) * 64 + lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int h = KVH ? r >> 1 : dt >> 2, e = KVH ? 8 * (r & 1) + dt : 4 * r + (dt & 3);
        o[h][e] = __fdiv_rn(O[r], L);
        top[h] = max(top[h], __float_as_uint(fabsf(o[h][e])));
      }
    }
    if constexpr (KVH) {
      top[0] = top[1] = max(top[0], top[1]);
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) top[h] = max(top[h], lane_xor<16>(top[h]));
    }
    if (orow >= A.S) return;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float amax = __uint_as_float(top[h]);
      const float id = amax != 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
      uint32_t word[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        word[i] = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) word[i] |= (uint32_t)(uint8_t)(int8_t)rintf(__fmul_rn(o[h][4 * i + e], id)) << (8 * e);
      }
      const int at = ooff + (KVH ? 32 * g + 16 * h : 64 * h + 16 * g);
      *(uint4*)(A.ocodes + q8_rows_code(A.S, orow, at / 16)) = make_uint4(word[0], word[1], word[2], word[3]);
      if (KVH ? h == 0 : (g & 1) == 0) A.oscales[q8_rows_scale(A.S, orow, at / 32)] = __half2float(__float2half_rn(__fdiv_rn(amax, 127.0f)));
    }
  } else {
    if (orow >= A.S) return;
    const int d0 = (wave >> 1) * (NDT / 2);  // half of the dt tiles per wave
    float* dst = A.out + (size_t)orow * A.out_stride + ooff;
    float o[NDT / 2][4];
#pragma unroll
    for (int dt = 0; dt < NDT / 2; ++dt) {
      const v4f O = box[(u * NDT + d0 + dt) * 64 + lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) o[dt][r] = __fdiv_rn(O[r], L);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 4 * g + r;
      float* run = dst + (KVH ? 8 * i + d0 : 64 * (d0 / 4) + 4 * i + d0 % 4);
      if constexpr (NDT == 8)
        *(v4f*)run = v4f{o[0][r], o[1][r], o[2][r], o[3][r]};
      else
        *(float2*)run = make_float2(o[0][r], o[1][r]);
    }
  }
}

}  // namespace dev
}  // namespace mtg
