// prefill_wt.hip - the block prefill for f16 and q4_K weights: the prompt rows go
// through the decoder in blocks of up to 2,048 rows with each weight matrix
// streamed once per block (Qwen3Decoder::prefill, src/qwen3_decoder.cpp:162-166),
// as prefill.hip does for q8_0. Per layer:
//   k_pf_act_wt     RMSNorm * gain (or the rows as they are) and the weight type's
//                   vec_dot_type: f16 values, or q8_K blocks (quantize_row_q8_K)
//   k_pf_gemm_f16   f16 (f32) weights x f16 (f32) activations on f32 MFMA, in the canonical
//                   segment order (below)
//   k_pf_gemm_q4k   q4_K weights x q8_K activations: exact int32 sums per
//                   superblock on int8 MFMA, the float chain over superblocks
// with prefill.hip's q/k norm + RoPE + KV append and causal attention (its f32
// output variant) in between. Outputs equal the oracle's and the verify path's
// bit for bit (the same orders as the per-op kernels of kernels_wt.hip).
#include <type_traits>

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "device_common.hpp"

namespace mtg {
namespace {
using namespace dev;

// ---------------------------------------------------------- activations ----
// Grid (S rows, K / 256), 256 threads, one element per thread: the arithmetic of
// k_act_f16 / k_act_q8k for any number of rows. gain == nullptr: no norm.
template <int WT>
__global__ void __launch_bounds__(256)
k_pf_act_wt(const float* __restrict__ src, int S, int K, const float* __restrict__ gain, float eps,
            uint16_t* __restrict__ f16_out, ActQ8K a, float* __restrict__ f32_out) {
  const int t = blockIdx.x, b = blockIdx.y, k = b * 256 + threadIdx.x;
  if (t >= S) return;
  const float* xr = src + (size_t)t * K;
  __shared__ float s_scale;
  float y = xr[k];
  const float gk = gain ? gain[k] : 0.0f;
  if (gain) {
    if (threadIdx.x < 64) {
      const float sc = row_rms_scale(xr, K, eps);
      if (threadIdx.x == 0) s_scale = sc;
    }
    __syncthreads();
    y = __fmul_rn(__fmul_rn(y, s_scale), gk);
  }
  if constexpr (WT == MTG_TYPE_F16) {
    f16_out[(size_t)t * K + k] = __half_as_ushort(__float2half_rn(y));  // vec_dot_type F16
  } else if constexpr (WT == MTG_TYPE_F32) {
    f32_out[(size_t)t * K + k] = y;  // vec_dot_type F32: the row as it is
  } else {
    q8k_block256(y, a, t, K, b);
  }
}

// The rows of the output tile that this lane holds (the MFMA result layout:
// lane (n, g) = (lane % 16, lane / 16) holds weight rows 4 g + r, r < 4, of the
// wave's 16, for activation row n of the column tile), after the epilogue
// (epi: store, residual add, or the encoder's linear = mul_mat + bias, then GELU,
// SiLU or the residual add; the SwiGLU is applied before this).
// n0: the first of the 4 weight rows in the output's row space.
__device__ __forceinline__ void pf_store4(int epi, float* out, int N, int t, int n0, const float (&v)[4],
                                          const float* bias) {
  float* dst = out + (size_t)t * N + n0;
  float y[4] = {v[0], v[1], v[2], v[3]};
  if (epi >= PF_EPI_BIAS) {
    const v4f b = *(const v4f*)(bias + n0);
#pragma unroll
    for (int q = 0; q < 4; ++q) y[q] = __fadd_rn(y[q], b[q]);
    if (epi == PF_EPI_BIAS_GELU) {
      dev_gelu_erf_n<4>(y);
    } else if (epi == PF_EPI_BIAS_SILU) {
#pragma unroll
      for (int q = 0; q < 4; ++q) y[q] = dev_silu(y[q]);
    }
  }
  v4f o;
  if (epi == PF_EPI_RESID || epi == PF_EPI_BIAS_RESID) {
    const v4f x = *(const v4f*)dst;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = __fadd_rn(x[q], y[q]);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = y[q];
  }
  *(v4f*)dst = o;
}

// ------------------------------------------------------- f16 / f32 GEMM ----
// out[s][n] in the canonical f16 dot (the oracle's mul_mat_f16, the per-op k_gemm_f16):
// K in 64 consecutive segments of L = K / 64 elements, each an fma chain from 0 over
// its elements in order (a product of two f16 values is exact in f32), the 64 partials
// reduced by the xor butterfly (v[i] + v[i ^ 32], then 16, .. 1, lane 0).
// v_mfma_f32_16x16x4f32 returns fma(a3, b3, fma(a2, b2, fma(a1, b1, fma(a0, b0, c))))
// per output, so L / 4 chained MFMAs from a zero accumulator are one segment's chain
// (k-step s: elements 4 s + kk held by lane group kk). The segments run in 6-bit
// bit-reversed order: the butterfly's tree is then the balanced binary tree over the
// run, folded as it goes with a stack of partials (a binary counter).
// F32: f32 weights and activations (vec_dot_type F32), the same segments, chains and
// tree: each step of a segment's chain is one fma of two f32 values, as the oracle's
// mul_mat_f32 and the per-op k_gemm_f32 take it.
//
// What bounds it: f32 MFMAs (33 cycles each) and every vector instruction beside them,
// which do not overlap: 420 us per decoder layer of 2,048 rows for the MFMAs alone. So a
// wave takes 32 weight rows x 32 activation rows (four chains; one 16-byte LDS read
// feeds four k-steps of two of them), 64 elements of the rows are staged per barrier,
// converted once per workgroup, the next 64 in flight in registers, and the first tree
// levels, those inside a stage, are plain sums. NW waves: 16 NW weight rows x 64
// activation rows; 8 where that leaves every CU a workgroup (its loads per MFMA are
// three quarters of 4's), else 4.
// Per layer of 2,048 rows, f16: q|k|v 237 -> 173 us, gate/up 345 -> 261, o 114 -> 85, down
// 165 -> 130 (before: 16 x 64 tiles per wave, one 4-byte LDS read per operand and MFMA, a
// barrier and a six-level fold per segment).
__device__ __forceinline__ int bitrev6(int k) { return (int)(__builtin_bitreverse32((uint32_t)k) >> 26); }

template <int L, int NW>
struct PfF16 {
  static constexpr int LPS = L == 16 ? 4 : L == 32 ? 2 : 1;  // segments per stage
  static constexpr int LV = LPS == 4 ? 2 : LPS == 2 ? 1 : 0;  // their tree levels
  static constexpr int rows = 16 * NW + 64, stride = L + 4;    // staged rows; floats per row (bank spread)
  static constexpr int leaf = rows * stride, stage = LPS * leaf;
  static constexpr size_t bytes = (size_t)2 * stage * 4;
};

template <bool GLU, int L, bool F32, int NW>
__global__ void __launch_bounds__(64 * NW, 2)
k_pf_gemm_f16(const void* __restrict__ wv, const void* __restrict__ w2v, int N, const void* __restrict__ xv, int S,
              float* __restrict__ out, int epi, const float* __restrict__ bias) {
  using P = PfF16<L, NW>;
  using E = typename std::conditional<F32, float, uint16_t>::type;
  constexpr int EP = 16 / (int)sizeof(E);  // elements per 16-byte piece
  constexpr int K = 64 * L, NP = L / EP, WR = 16 * NW, GR = WR / 2;  // pieces per row and segment; weight rows; gate rows
  constexpr int NPIECE = P::LPS * P::rows * NP, PPT = (NPIECE + 64 * NW - 1) / (64 * NW);
  extern __shared__ v4f pf16_lds_v4[];
  float* const s_st = (float*)pf16_lds_v4;
  const E* w = (const E*)wv;
  const E* w2 = (const E*)w2v;
  const E* x = (const E*)xv;
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, kk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = wave >> 1, ws = wave & 1;
  const int s0 = blockIdx.y * 64;
  // staged row r: weight rows first (GLU: gate, then up), then the activation's 64;
  // rows past the matrix or the block read the last one, their outputs are dropped
  const int nrow = GLU ? GR * (int)blockIdx.x : WR * (int)blockIdx.x;
  auto row_of = [&](int r) -> const E* {
    if (r >= WR) return x + (size_t)min(s0 + r - WR, S - 1) * K;
    if constexpr (GLU) return (r < GR ? w : w2) + (size_t)min(nrow + r % GR, N - 1) * K;
    return w + (size_t)min(nrow + r, N - 1) * K;
  };
  const E* src[PPT];
  int dst[PPT], leaf[PPT];
#pragma unroll
  for (int i = 0; i < PPT; ++i) {
    const int p = min(tid + 64 * NW * i, NPIECE - 1), q = p / NP, j = p % NP, r = q % P::rows;
    leaf[i] = q / P::rows;
    src[i] = row_of(r) + EP * j;
    dst[i] = leaf[i] * P::leaf + r * P::stride + (EP / 4) * j;  // element 4 s + e of the segment at e * L / 4 + s
  }
  uint4 reg[PPT];
  auto fetch = [&](int st) {
#pragma unroll
    for (int i = 0; i < PPT; ++i) reg[i] = *(const uint4*)(src[i] + bitrev6(P::LPS * st + leaf[i]) * L);
  };
  auto stage = [&](float* buf) {
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      if (NPIECE % (64 * NW) && tid + 64 * NW * i >= NPIECE) continue;
      float* d = buf + dst[i];
      const uint32_t u[4] = {reg[i].x, reg[i].y, reg[i].z, reg[i].w};
      if constexpr (F32) {
#pragma unroll
        for (int e = 0; e < 4; ++e) d[e * (L / 4)] = __uint_as_float(u[e]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int sh = 16 * (e & 1);
          *(float2*)(d + e * (L / 4)) = make_float2(half_bits_to_float((uint16_t)(u[e / 2] >> sh)),
                                                    half_bits_to_float((uint16_t)(u[2 + e / 2] >> sh)));
        }
      }
    }
  };
  v4f stk[6 - P::LV][4];  // tile 2 a + b: weight rows 16 a, activation rows 16 b of the wave's 32 x 32
  v4f res[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    res[c] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int lvl = 0; lvl < 6 - P::LV; ++lvl) stk[lvl][c] = res[c];
  }
  auto add = [](v4f (&a)[4], const v4f (&b)[4]) {  // a = b + a, per output
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q) a[c][q] = __fadd_rn(b[c][q], a[c][q]);
  };
  const int aoff = (32 * wn + m) * P::stride + kk * (L / 4), boff = (WR + 32 * ws + m) * P::stride + kk * (L / 4);
  auto segment = [&](const float* lf, v4f (&cur)[4]) {
#pragma unroll
    for (int c = 0; c < 4; ++c) cur[c] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < L / 16; ++q) {
      v4f a[2], b[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        a[h] = *(const v4f*)(lf + aoff + 16 * h * P::stride + 4 * q);
        b[h] = *(const v4f*)(lf + boff + 16 * h * P::stride + 4 * q);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          cur[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[c >> 1][e], b[c & 1][e], cur[c], 0, 0, 0);
    }
  };
  fetch(0);
  stage(s_st);
  constexpr int NST = 64 / P::LPS;
  for (int st = 0; st < NST; ++st) {
    const float* buf = s_st + (st & 1) * P::stage;
    if (st + 1 < NST) fetch(st + 1);
    __syncthreads();  // stage st is complete; the other buffer's readers (stage st - 1) are done
    v4f cur[4];
    segment(buf, cur);
    if constexpr (P::LPS >= 2) {
      v4f nxt[4];
      segment(buf + P::leaf, nxt);
      add(cur, nxt);
    }
    if constexpr (P::LPS == 4) {
      v4f c2[4], c3[4];
      segment(buf + 2 * P::leaf, c2);
      segment(buf + 3 * P::leaf, c3);
      add(c2, c3);
      add(cur, c2);
    }
    // fold: while bit lvl of st is set, the left sibling (the earlier subtree) is added;
    // the first clear bit keeps the partial
    bool carry = true;
#pragma unroll
    for (int lvl = 0; lvl < 6 - P::LV; ++lvl) {
      if (carry) {
        if ((st >> lvl) & 1) {
          add(cur, stk[lvl]);
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c) stk[lvl][c] = cur[c];
          carry = false;
        }
      }
    }
    if (carry) {  // the last stage: the root
#pragma unroll
      for (int c = 0; c < 4; ++c) res[c] = cur[c];
    }
    if (st + 1 < NST) stage(s_st + ((st + 1) & 1) * P::stage);
  }
  if constexpr (GLU) {
    // the up waves hand their values to the gate waves of the same rows
    __syncthreads();
    float* s_up = s_st;  // [NW / 2 waves][4 tiles][64 lanes][4]
    constexpr int GW = NW / 4;
    if (wn >= GW)
#pragma unroll
      for (int c = 0; c < 4; ++c) *(v4f*)(s_up + (((wave - 2 * GW) * 4 + c) * 64 + lane) * 4) = res[c];
    __syncthreads();
    if (wn >= GW) return;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const v4f u = *(const v4f*)(s_up + ((wave * 4 + c) * 64 + lane) * 4);
#pragma unroll
      for (int q = 0; q < 4; ++q) res[c][q] = dev_swiglu(res[c][q], u[q]);
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int t = s0 + 32 * ws + 16 * (c & 1) + m, n = nrow + 32 * wn + 16 * (c >> 1) + 4 * kk;
    if (t >= S || n >= N) continue;
    const float v[4] = {res[c][0], res[c][1], res[c][2], res[c][3]};
    pf_store4(GLU ? (int)PF_EPI_STORE : epi, out, N, t, n, v, bias);
  }
}

// ------------------------------------------------------------ q4_K GEMM ----
// 64 weight rows x 64 activation rows per workgroup (the same wave roles as
// k_pf_gemm_f16). Per superblock of 256: the activation codes and scales of the
// 64 rows are staged in LDS (row stride 288 bytes: a wave's 8-byte operand reads
// take the minimum two passes), the next superblock's in flight in registers with
// the wave's weight bytes. For each 16 x 16 output tile the exact int32 sums
// dot = sum_j sc_j * sub_j (the 6-bit scale split as 8 * (sc >> 3) + (sc & 7): two
// int8 MFMA accumulators of nibble * factor <= 105) and mins = sum_j mn_j * sum(x_j)
// come from v_mfma_i32_16x16x32_i8 (the per-op k_gemm_q4m's sums), then the
// oracle's chain over superblocks in order: acc = (acc + (d_w d_x) dot) -
// (dmin_w d_x) mins.
constexpr int kQ4RowStride = 288;

template <bool GLU>
__global__ void __launch_bounds__(256)
k_pf_gemm_q4k(const uint8_t* __restrict__ w, const uint8_t* __restrict__ w2, int N, int K, ActQ8K a, int S,
              float* __restrict__ out, int epi, const float* __restrict__ bias) {
  __shared__ __align__(16) int8_t s_q[2][64 * kQ4RowStride];
  __shared__ float s_dx[2][64];
  __shared__ float s_dw[4][16 * 2];  // per wave: d, dmin of its 16 weight rows
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, row = lane & 15, g = lane >> 4;
  const int NB = K / 256, s0 = blockIdx.y * 64;
  const uint8_t* wr = GLU ? (wave < 2 ? w : w2) + (size_t)(32 * blockIdx.x + 16 * (wave & 1) + row) * NB * 144
                          : w + (size_t)(64 * blockIdx.x + 16 * wave + row) * NB * 144;
  // staging: thread tid takes 16-byte pieces tid + 256 i (i < 4) of the 64 x 256
  // code block (row p / 16, bytes 16 (p % 16) ..); threads < 64 a row's scale
  uint4 nq[4];
  float ndx = 0.0f;
  uint2 nw[4];
  v4i nh;
  auto fetch = [&](int b) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = tid + 256 * i, r = p >> 4, c = p & 15;
      nq[i] = s0 + r < S ? *(const uint4*)(a.qs + (size_t)(s0 + r) * K + b * 256 + 16 * c) : make_uint4(0, 0, 0, 0);
    }
    if (tid < 64) ndx = s0 + tid < S ? a.d[(size_t)(s0 + tid) * NB + b] : 0.0f;
#pragma unroll
    for (int mm = 0; mm < 4; ++mm) nw[mm] = *(const uint2*)(wr + b * 144 + 16 + 32 * mm + 8 * g);
    nh = *(const v4i*)(wr + b * 144);
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = tid + 256 * i, r = p >> 4, c = p & 15;
      *(uint4*)(s_q[buf] + r * kQ4RowStride + 16 * c) = nq[i];
    }
    if (tid < 64) s_dx[buf][tid] = ndx;
  };
  float res[4][4];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct)
#pragma unroll
    for (int r = 0; r < 4; ++r) res[ct][r] = 0.0f;
  fetch(0);
  stage(0);
  for (int b = 0; b < NB; ++b) {
    const int buf = b & 1;
    const uint2 qw[4] = {nw[0], nw[1], nw[2], nw[3]};
    const v4i h = nh;
    if (b + 1 < NB) fetch(b + 1);
    __syncthreads();  // superblock b is staged; the other buffer's readers are done
    int sc[8], mn[8];
    q4k_scales_w((uint32_t)h[1], (uint32_t)h[2], (uint32_t)h[3], sc, mn);
    // d, dmin of the wave's rows through its LDS slot (lanes 0..15 own them; LDS
    // accesses of a wave execute in order)
    if (g == 0) {
      s_dw[wave][row * 2] = half_bits_to_float((uint16_t)((uint32_t)h[0] & 0xffffu));
      s_dw[wave][row * 2 + 1] = half_bits_to_float((uint16_t)((uint32_t)h[0] >> 16));
    }
    float dw[4], dmw[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      dw[r] = s_dw[wave][(4 * g + r) * 2];
      dmw[r] = s_dw[wave][(4 * g + r) * 2 + 1];
    }
    // the A operands of the 8 sub-blocks: nibbles x (sc >> 3), x (sc & 7), and mn
    long ah[8], al[8], am[8];
#pragma unroll
    for (int mm = 0; mm < 4; ++mm)
#pragma unroll
      for (int hi = 0; hi < 2; ++hi) {
        const int s = 2 * mm + hi;
        const uint32_t q0 = hi ? (qw[mm].x >> 4) & 0x0F0F0F0Fu : qw[mm].x & 0x0F0F0F0Fu;
        const uint32_t q1 = hi ? (qw[mm].y >> 4) & 0x0F0F0F0Fu : qw[mm].y & 0x0F0F0F0Fu;
        const uint32_t fh = (uint32_t)(sc[s] >> 3), fl = (uint32_t)(sc[s] & 7), fm = (uint32_t)mn[s] * 0x01010101u;
        ah[s] = (long)(((uint64_t)(q1 * fh) << 32) | (q0 * fh));
        al[s] = (long)(((uint64_t)(q1 * fl) << 32) | (q0 * fl));
        am[s] = (long)(((uint64_t)fm << 32) | fm);
      }
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      v4i ahi = {0, 0, 0, 0}, alo = {0, 0, 0, 0}, amn = {0, 0, 0, 0};
      const int8_t* xb = s_q[buf] + (16 * ct + row) * kQ4RowStride + 8 * g;
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const long bv = *(const long*)(xb + 32 * s);
        ahi = __builtin_amdgcn_mfma_i32_16x16x32_i8(ah[s], bv, ahi, 0, 0, 0);
        alo = __builtin_amdgcn_mfma_i32_16x16x32_i8(al[s], bv, alo, 0, 0, 0);
        amn = __builtin_amdgcn_mfma_i32_16x16x32_i8(am[s], bv, amn, 0, 0, 0);
      }
      const float dx = s_dx[buf][16 * ct + row];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int dot = 8 * ahi[r] + alo[r];
        const float dm = __fmul_rn(dw[r], dx), dmin = __fmul_rn(dmw[r], dx);
        res[ct][r] = __fadd_rn(res[ct][r], __fmul_rn(dm, (float)dot));
        res[ct][r] = __fsub_rn(res[ct][r], __fmul_rn(dmin, (float)amn[r]));
      }
    }
    if (b + 1 < NB) stage(buf ^ 1);
  }
  if constexpr (GLU) {
    __syncthreads();
    float* s_up = (float*)s_q[0];  // [2 tiles][4 ct][64 lanes][4]
    if (wave >= 2)
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
        *(v4f*)(s_up + (((wave & 1) * 4 + ct) * 64 + lane) * 4) = v4f{res[ct][0], res[ct][1], res[ct][2], res[ct][3]};
    __syncthreads();
    if (wave >= 2) return;
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      const int t = s0 + 16 * ct + row;
      if (t >= S) continue;
      const v4f u = *(const v4f*)(s_up + (((wave & 1) * 4 + ct) * 64 + lane) * 4);
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = dev_swiglu(res[ct][q], u[q]);
      pf_store4(PF_EPI_STORE, out, N, t, 32 * blockIdx.x + 16 * (wave & 1) + 4 * g, v, nullptr);
    }
  } else {
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      const int t = s0 + 16 * ct + row;
      if (t >= S) continue;
      pf_store4(epi, out, N, t, 64 * blockIdx.x + 16 * wave + 4 * g, res[ct], bias);
    }
  }
}

}  // namespace

// ================================================================ launches ==
void launch_pf_act_wt(hipStream_t s, int wtype, const float* src, int S, int K, const float* gain, float eps,
                      const WtAct& act) {
  const dim3 grid((unsigned)S, (unsigned)(K / 256));
  if (wtype == MTG_TYPE_F16)
    hipLaunchKernelGGL(k_pf_act_wt<MTG_TYPE_F16>, grid, dim3(256), 0, s, src, S, K, gain, eps, act.f16h, act.q8k,
                       act.f32);
  else if (wtype == MTG_TYPE_F32)
    hipLaunchKernelGGL(k_pf_act_wt<MTG_TYPE_F32>, grid, dim3(256), 0, s, src, S, K, gain, eps, act.f16h, act.q8k,
                       act.f32);
  else
    hipLaunchKernelGGL(k_pf_act_wt<MTG_TYPE_Q4_K>, grid, dim3(256), 0, s, src, S, K, gain, eps, act.f16h, act.q8k,
                       act.f32);
}

void launch_pf_gemm_wt(hipStream_t s, int wtype, int epi, const uint8_t* w, const uint8_t* w2, int N, int K,
                       const WtAct& act, int S, float* out, const float* bias) {
  const bool glu = epi == PF_EPI_SWIGLU;
  const dim3 grid((unsigned)(glu ? N / 32 : N / 64), (unsigned)((S + 63) / 64));
  if (wtype == MTG_TYPE_Q4_K) {
    if (glu)
      hipLaunchKernelGGL(k_pf_gemm_q4k<true>, grid, dim3(256), 0, s, w, w2, N, K, act.q8k, S, out, epi, bias);
    else
      hipLaunchKernelGGL(k_pf_gemm_q4k<false>, grid, dim3(256), 0, s, w, w2, N, K, act.q8k, S, out, epi, bias);
    return;
  }
  const bool f32 = wtype == MTG_TYPE_F32;
  const void* xa = f32 ? (const void*)act.f32 : (const void*)act.f16h;
  // eight waves (128 weight rows) once every CU gets a workgroup, else four: N 1,024, K 3,072,
  // 2,048 rows 130 us with 256 workgroups of eight, 1,819 rows 130 us with 464 of four
  const int wide_n = glu ? N / 64 : N / 128;
  const bool wide = (size_t)wide_n * grid.y >= 256;
  const dim3 wgrid((unsigned)((glu ? 2 * N : N) + 127) / 128, grid.y);
#define MTG_PF_F16_W(G, L, F, NW, GRID) \
  hipLaunchKernelGGL((k_pf_gemm_f16<G, L, F, NW>), GRID, dim3(64 * NW), (PfF16<L, NW>::bytes), s, w, w2, N, xa, S, out, epi, bias)
#define MTG_PF_F16(G, L)                             \
  do {                                               \
    if (f32 && wide) MTG_PF_F16_W(G, L, true, 8, wgrid);  \
    else if (f32) MTG_PF_F16_W(G, L, true, 4, grid);      \
    else if (wide) MTG_PF_F16_W(G, L, false, 8, wgrid);   \
    else MTG_PF_F16_W(G, L, false, 4, grid);              \
  } while (0)
#define MTG_PF_F16_K(G)                        \
  switch (K) {                                 \
    case 1024: MTG_PF_F16(G, 16); break;       \
    case 2048: MTG_PF_F16(G, 32); break;       \
    case 3072: MTG_PF_F16(G, 48); break;       \
    default: MTG_PF_F16(G, 64); break;         \
  }
  if (glu) { MTG_PF_F16_K(true); }
  else { MTG_PF_F16_K(false); }
#undef MTG_PF_F16_K
#undef MTG_PF_F16
#undef MTG_PF_F16_W
}

hipError_t prepare_kernels_pf_wt() {
  hipError_t e = hipSuccess;
#define MTG_PF_LDS(G, L, F)                                                                                      \
  if (e == hipSuccess)                                                                                           \
    e = hipFuncSetAttribute((const void*)k_pf_gemm_f16<G, L, F, 8>, hipFuncAttributeMaxDynamicSharedMemorySize,  \
                            (int)PfF16<L, 8>::bytes);                                                            \
  if (e == hipSuccess)                                                                                           \
    e = hipFuncSetAttribute((const void*)k_pf_gemm_f16<G, L, F, 4>, hipFuncAttributeMaxDynamicSharedMemorySize,  \
                            (int)PfF16<L, 4>::bytes);
#define MTG_PF_LDS_K(G, F) MTG_PF_LDS(G, 16, F) MTG_PF_LDS(G, 32, F) MTG_PF_LDS(G, 48, F) MTG_PF_LDS(G, 64, F)
  MTG_PF_LDS_K(false, false)
  MTG_PF_LDS_K(false, true)
  MTG_PF_LDS_K(true, false)
  MTG_PF_LDS_K(true, true)
#undef MTG_PF_LDS_K
#undef MTG_PF_LDS
  return e;
}

int pf_gemm_wt_supported(int wtype, int K) {
  if (wtype == MTG_TYPE_Q4_K) return K % 256 == 0;
  return K == 1024 || K == 2048 || K == 3072 || K == 4096;
}

}  // namespace mtg
