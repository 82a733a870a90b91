// prefill.hip - the prompt prefill on the device: S rows through the decoder
// with each weight matrix streamed once per block of rows (Qwen3Decoder::prefill,
// src/qwen3_decoder.cpp:162-166, which runs the fused prompt as one batch).
//
// The verify path processes at most 16 rows per weight pass; a 1,600-row prompt
// through it costs 100 full weight streams. Here every layer is a short
// sequence of kernels over all rows of a block (up to kPfRows):
//   k_pf_norm_quant  RMSNorm * gain and the q8_0 activation conversion, codes and
//                    scales (f16 values) in the GEMM's order (q8_rows_code)
//   k_pf_gemm        q8_0 weight tiles x activation rows on v_mfma_i32_32x32x32_i8
//                    (one exact int32 dot per block), epilogue store / residual
//                    add / SwiGLU
//   k_pf_quant       q8_0 conversion of f32 rows (the SwiGLU output)
//   k_pf_qk_rope     q/k RMSNorm + NEOX RoPE, K/V written into the cache
//   k_attn_block     causal attention on f32 MFMA (attn_block.hpp), writing the
//                    o-projection's q8_0 activation
// Every reduction follows the canonical order of device_common.hpp, so hidden
// rows and the KV cache equal the verify path's and the oracle's bit for bit:
//   * GEMM: per output, 4 K-slices of block pairs, even / odd fma chains per
//     slice in block order, ((s0 + s1) + s2) + s3 per parity, then even + odd;
//   * attention: attn_block.hpp, the same chunk terms and merge chain the verify
//     path runs.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "attn_block.hpp"
#include "device_common.hpp"

namespace mtg {
namespace {
using namespace dev;

constexpr int kH = 1024;         // hidden (the RMSNorm partials assume 1024)

// ---------------------------------------------------------- activations ----
// One wave per row of 1024: lane l holds elements 16 l .. 16 l + 15 (the
// canonical RMSNorm partials); q8_0 blocks are lanes (2 b, 2 b + 1).
__global__ void __launch_bounds__(256)
k_pf_norm_quant(const float* __restrict__ src, int S, const float* __restrict__ gain, float eps,
                int8_t* __restrict__ codes, float* __restrict__ scales, float* __restrict__ normed_out) {
  const int row = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= S) return;
  const float* xr = src + (size_t)row * kH + 16 * lane;
  float v[16];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const v4f q = *(const v4f*)(xr + 4 * i);
    v[4 * i] = q[0];
    v[4 * i + 1] = q[1];
    v[4 * i + 2] = q[2];
    v[4 * i + 3] = q[3];
  }
  double s = 0.0;
#pragma unroll
  for (int e = 0; e < 16; ++e) s += (double)__fmul_rn(v[e], v[e]);
  s = wave_sum_d(s);
  const float scale = dev_rms_scale((float)(s / (double)kH), eps);
  float y[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) y[e] = __fmul_rn(__fmul_rn(v[e], scale), gain[16 * lane + e]);
  if (normed_out) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const v4f o = {y[4 * i], y[4 * i + 1], y[4 * i + 2], y[4 * i + 3]};
      *(v4f*)(normed_out + (size_t)row * kH + 16 * lane + 4 * i) = o;
    }
  }
  float amax = 0.0f;
#pragma unroll
  for (int e = 0; e < 16; ++e) amax = fmaxf(amax, fabsf(y[e]));
  amax = __uint_as_float(max(__float_as_uint(amax), dpp_u<kDppQuadXor1>(__float_as_uint(amax))));
  const float d = __fdiv_rn(amax, 127.0f);
  const float id = amax != 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
  uint32_t packed[4];
#pragma unroll
  for (int w4 = 0; w4 < 4; ++w4) {
    uint32_t u = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) u |= (uint32_t)(uint8_t)(int8_t)rintf(__fmul_rn(y[4 * w4 + b], id)) << (8 * b);
    packed[w4] = u;
  }
  *(uint4*)(codes + q8_rows_code(S, row, lane)) = make_uint4(packed[0], packed[1], packed[2], packed[3]);
  if ((lane & 1) == 0) scales[q8_rows_scale(S, row, lane / 2)] = __half2float(__float2half_rn(d));
}

// q8_0 conversion of f32 rows of K (a multiple of 32): one wave per row, lane =
// one 32-element block at a time.
__global__ void __launch_bounds__(256)
k_pf_quant(const float* __restrict__ src, int S, int K, int8_t* __restrict__ codes, float* __restrict__ scales) {
  const int row = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= S) return;
  for (int b = lane; b < K / 32; b += 64) {
    const float* xr = src + (size_t)row * K + 32 * b;
    float v[32];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const v4f q = *(const v4f*)(xr + 4 * i);
      v[4 * i] = q[0];
      v[4 * i + 1] = q[1];
      v[4 * i + 2] = q[2];
      v[4 * i + 3] = q[3];
    }
    float amax = 0.0f;
#pragma unroll
    for (int e = 0; e < 32; ++e) amax = fmaxf(amax, fabsf(v[e]));
    const float d = __fdiv_rn(amax, 127.0f);
    const float id = amax != 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
    uint32_t packed[8];
#pragma unroll
    for (int w4 = 0; w4 < 8; ++w4) {
      uint32_t u = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) u |= (uint32_t)(uint8_t)(int8_t)rintf(__fmul_rn(v[4 * w4 + e], id)) << (8 * e);
      packed[w4] = u;
    }
    *(uint4*)(codes + q8_rows_code(S, row, 2 * b)) = make_uint4(packed[0], packed[1], packed[2], packed[3]);
    *(uint4*)(codes + q8_rows_code(S, row, 2 * b + 1)) = make_uint4(packed[4], packed[5], packed[6], packed[7]);
    scales[q8_rows_scale(S, row, b)] = __half2float(__float2half_rn(d));
  }
}

// ----------------------------------------------------------------- GEMM ----
// out[s][n] = the canonical q8_0 dot of weight row n and activation row s: per
// 32-block the exact int32 sum (v_mfma_i32_32x32x32_i8), then one fma of it with
// dw * dx (exact in f32) into the even or odd chain of the K-slice; slices add
// ((s0 + s1) + s2) + s3 per parity, then even + odd.
//
// What bounds it: those float steps. Every output needs a conversion, a product
// and an fma per block, 48 vector instructions per 32 x 32 block of outputs (196
// cycles with the MFMA's 35 beside them), 61 us per decoder layer at 1,600 rows. So
// a wave keeps a 32 x 32 tile's running sums in registers and nothing else is vector
// work: both operands lie in memory in the order the MFMA takes them and go straight
// to LDS, several 64-element steps ahead of their use. A workgroup takes 64 activation
// rows x 64 weight rows (SwiGLU: 32 of gate and the same 32 of up).
enum { PF_STORE = 0, PF_RESID = 1, PF_SWIGLU = 2, PF_BIAS = 3, PF_BIAS_GELU = 4, PF_BIAS_SILU = 5, PF_BIAS_RESID = 6 };
typedef int v16i __attribute__((ext_vector_type(16)));

// 16 (4) bytes per lane from memory to LDS at lds + 16 (4) * lane, counted in vmcnt.
// lds is a byte address, uniform over the wave. m0 is the compiler's own for indexed
// access: named, so that no value of its is taken to outlive the statement (the warning
// about a reserved register says that it is not saved around it, which nothing needs).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_fill16(const void* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void lds_fill4(const void* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop

// One 64-element step in LDS: the codes of 4 weight units, then 4 parts x 64 rows x 16
// bytes of the activation, the units' scales (4 x 32 f16), [parity][64 rows] f32 scales.
struct PgStage {
  static constexpr int codes = 4096, wscales = 8192, dx = 8448, bytes = 8960, fills = 3;
};

// ST: stages in flight. The workgroups of an XCD walk K together, so that a step is new
// to its L2 for all of them. Four stages let four workgroups share a CU; a grid of 512
// or fewer has at most two per CU and takes eight (1,600 rows: K 2,048 / 3,072, N 1,024,
// 400 workgroups: 28 / 41.6 us with four, 25 / 36.6 with eight; gate and up, 2,400:
// 50 and 65). Per layer at 1,600 rows: q|k|v 63 -> 33 us, gate/up 95 -> 50, o 33 -> 25,
// down 48 -> 37 (before: codes staged through registers, one barrier per step with its
// loads just ahead, block-diagonal 16 x 16 MFMAs).
// Four workgroups leave a wave 128 registers: enough but for GELU's doubles (<4, 4>: 9 of
// the running totals are spilled, moved once per K-slice).
template <int EPI, int ST>
__global__ void __launch_bounds__(256, ST == 4 ? 4 : 2)
k_pf_gemm(const uint8_t* __restrict__ w, const uint8_t* __restrict__ w2, int N, int K,
          const int8_t* __restrict__ codes, const float* __restrict__ scales, int S, float* __restrict__ out,
          const float* __restrict__ bias) {
  constexpr bool GLU = EPI == PF_SWIGLU;
  __shared__ __align__(16) uint8_t s_st[ST * PgStage::bytes];
  const int tid = threadIdx.x, lane = tid & 63, j = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s0 = blockIdx.y * 64, rb = gridDim.y, bps = K / kPairK;
  const int ws = wave & 1, wn = wave >> 1;  // the wave's 32 rows, its 32 weight rows (GLU: gate or up)
  // fills: wave w brings weight unit w, part w of the codes, and the weight scales
  // (waves 0, 1: half each) or the activation scales of parity w - 2
  auto unit_of = [&](int u) {
    if constexpr (GLU) return (u < 2 ? w : w2) + (size_t)(2 * blockIdx.x + (u & 1)) * bps * kUnitBytes;
    return w + (size_t)(4 * blockIdx.x + u) * bps * kUnitBytes;
  };
  const uint8_t* wsrc = unit_of(wave) + 16 * lane;
  const int8_t* xsrc = codes + ((size_t)(s0 / 64) * 256 + 64 * wave + lane) * 16;
  const bool act_scale = wave >= 2;
  const uint8_t* dsrc = act_scale ? (const uint8_t*)(scales + (size_t)(wave & 1) * rb * 64 + s0 + lane)
                                  : unit_of(lane >> 4) + 1024 + 4 * (lane & 15);
  const size_t xstep = (size_t)rb * 4096, dstep = act_scale ? (size_t)rb * 512 : (size_t)kUnitBytes;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)s_st;
  const int ddst = act_scale ? PgStage::dx + 256 * (wave & 1) : PgStage::wscales;  // waves 0 and 1 bring the same bytes
  auto fill = [&](int bp) {  // past the last pair: the last one again, into a stage nobody reads
    const uint32_t st = lds0 + (bp % ST) * PgStage::bytes;
    const int at = min(bp, bps - 1);
    lds_fill16(wsrc + (size_t)at * kUnitBytes, st + wave * 1024);
    lds_fill16(xsrc + at * xstep, st + PgStage::codes + wave * 1024);
    lds_fill4(dsrc + at * dstep, st + ddst);
  };
  const int ut = 2 * wn + (j >> 4);  // lane j holds weight row j of 32, in this unit
  float part[2][16], tot[2][16];     // [parity][register]
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int r = 0; r < 16; ++r) part[p][r] = tot[p][r] = 0.0f;
  const v16i zero = {};
#pragma unroll
  for (int i = 0; i < ST - 1; ++i) fill(i);
#pragma unroll 1
  for (int sl = 0, bp = 0; sl < 4; ++sl) {
#pragma unroll 1
    for (const int end = bps * (sl + 1) / 4; bp < end; ++bp) {
      // this wave's fills of pair bp are done (those of later pairs may be in flight);
      // behind the barrier everyone's are, and nobody reads pair bp - 1 any more
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((ST - 2) * PgStage::fills) : "memory");
      fill(bp + ST - 1);
      const uint8_t* st = s_st + (bp % ST) * PgStage::bytes;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const v4i a = *(const v4i*)(st + PgStage::codes + (2 * p + h) * 1024 + 16 * (32 * ws + j));
        const v4i bw = *(const v4i*)(st + ut * 1024 + (2 * p + h) * 256 + 16 * (j & 15));
        const float dw = half_bits_to_float(*(const uint16_t*)(st + PgStage::wscales + ut * 64 + 2 * (16 * p + (j & 15))));
        const v16i c = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, bw, zero, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // registers 4 i + e: rows 8 i + 4 h + e
          const v4f dx = *(const v4f*)(st + PgStage::dx + 4 * (64 * p + 32 * ws + 8 * i + 4 * h));
#pragma unroll
          for (int e = 0; e < 4; ++e) part[p][4 * i + e] = fmaf((float)c[4 * i + e], dw * dx[e], part[p][4 * i + e]);
        }
      }
    }
    // a K-slice ends: fold it into the running total (0 + s0 is s0: no sum is -0)
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        tot[p][r] = __fadd_rn(tot[p][r], part[p][r]);
        part[p][r] = 0.0f;
      }
  }
  float y[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) y[r] = __fadd_rn(tot[0][r], tot[1][r]);  // even + odd
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no fill outlives the workgroup
  if constexpr (GLU) {
    // the up waves hand their values to the gate waves of the same rows
    __syncthreads();
    v4f* s_up = (v4f*)s_st + (ws * 64 + lane) * 4;
    if (wn == 1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) s_up[i] = v4f{y[4 * i], y[4 * i + 1], y[4 * i + 2], y[4 * i + 3]};
    }
    __syncthreads();
    if (wn == 1) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) y[r] = dev_swiglu(y[r], s_up[r / 4][r % 4]);
  }
  const int n = GLU ? 32 * (int)blockIdx.x + j : 64 * (int)blockIdx.x + 32 * wn + j;
  if constexpr (EPI >= PF_BIAS) {
    // linear = mul_mat + bias, then the activation or the residual add
    const float bn = bias[n];
#pragma unroll
    for (int r = 0; r < 16; ++r) y[r] = __fadd_rn(y[r], bn);
    if constexpr (EPI == PF_BIAS_GELU) {
#pragma unroll
      for (int r = 0; r < 16; r += 8) {
        float e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = y[r + i];
        dev_gelu_erf_n<8>(e);
#pragma unroll
        for (int i = 0; i < 8; ++i) y[r + i] = e[i];
      }
    }
    if constexpr (EPI == PF_BIAS_SILU)
#pragma unroll
      for (int r = 0; r < 16; ++r) y[r] = dev_silu(y[r]);
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = s0 + 32 * ws + 8 * (r / 4) + 4 * h + r % 4;
    if (row >= S) continue;
    float* dst = out + (size_t)row * N + n;
    *dst = (EPI == PF_RESID || EPI == PF_BIAS_RESID) ? __fadd_rn(*dst, y[r]) : y[r];
  }
}

// ------------------------------------------------- q/k norm, rope, append ---
// grid (S rows, n_heads + 2 n_kv_heads units), one wave per unit: the same
// arithmetic as the verify path's k_qk_rope_append at position past0 + row.
__global__ void __launch_bounds__(64)
k_pf_qk_rope(const float* __restrict__ qkv, int S, int past0, int n_heads, int n_kv_heads,
             const float* __restrict__ q_norm, const float* __restrict__ k_norm, float eps,
             const float* __restrict__ rope, float* __restrict__ q_out, KvLayer kv) {
  const int t = blockIdx.x;
  if (t >= S) return;
  const int u = blockIdx.y, i = threadIdx.x;
  const int QN = n_heads * kHeadDim, KN = n_kv_heads * kHeadDim, N = QN + 2 * KN;
  const int pos = past0 + t;
  const float* row = qkv + (size_t)t * N;
  const bool is_q = u < n_heads, is_k = !is_q && u < n_heads + n_kv_heads;
  const int col = is_q ? u * kHeadDim : is_k ? QN + (u - n_heads) * kHeadDim
                                             : QN + KN + (u - n_heads - n_kv_heads) * kHeadDim;
  float x0 = row[col + i], x1 = row[col + i + 64];
  if (is_q || is_k) {
    const float* gn = is_q ? q_norm : k_norm;
    double s = (double)__fmul_rn(x0, x0) + (double)__fmul_rn(x1, x1);
    s = wave_sum_d(s);
    const float scale = dev_rms_scale((float)(s / (double)kHeadDim), eps);
    const float y0 = __fmul_rn(__fmul_rn(x0, scale), gn[i]);
    const float y1 = __fmul_rn(__fmul_rn(x1, scale), gn[i + 64]);
    const float c = rope[(size_t)pos * kHeadDim + 2 * i], sn = rope[(size_t)pos * kHeadDim + 2 * i + 1];
    x0 = __fsub_rn(__fmul_rn(y0, c), __fmul_rn(y1, sn));
    x1 = __fadd_rn(__fmul_rn(y0, sn), __fmul_rn(y1, c));
  }
  if (is_q) {
    float* q = q_out + ((size_t)t * n_heads + u) * kHeadDim;
    q[i] = x0;
    q[i + 64] = x1;
    return;
  }
  const int h = is_k ? u - n_heads : u - n_heads - n_kv_heads;
  void* base = is_k ? kv.k : kv.v;
  const size_t off = ((size_t)h * kv.max_seq + pos) * kHeadDim;
  if (kv.f16) {
    __half* p = (__half*)base + off;
    p[i] = __float2half_rn(x0);
    p[i + 64] = __float2half_rn(x1);
  } else {
    float* p = (float*)base + off;
    p[i] = x0;
    p[i + 64] = x1;
  }
}

}  // namespace

// ================================================================ launches ==
// A kv head's rows in 32-bit byte offsets.
int pf_max_context() { return (int)(0x7fffffffu / (kHeadDim * 4)); }

void launch_pf_norm_quant(hipStream_t s, const float* src, int S, const float* gain, float eps, int8_t* codes,
                          float* scales, float* normed_out) {
  hipLaunchKernelGGL(k_pf_norm_quant, dim3((S + 3) / 4), dim3(256), 0, s, src, S, gain, eps, codes, scales,
                     normed_out);
}

void launch_pf_quant(hipStream_t s, const float* src, int S, int K, int8_t* codes, float* scales) {
  hipLaunchKernelGGL(k_pf_quant, dim3((S + 3) / 4), dim3(256), 0, s, src, S, K, codes, scales);
}

void launch_pf_gemm(hipStream_t s, int epi, const uint8_t* w, const uint8_t* w2, int N, int K, const int8_t* codes,
                    const float* scales, int S, float* out, const float* bias) {
  const dim3 blocks((unsigned)(epi == PF_SWIGLU ? N / 32 : N / 64), (unsigned)((S + 63) / 64));
  const bool deep = (size_t)blocks.x * blocks.y <= 512;  // two workgroups per CU or fewer
#define MTG_PF_GEMM(E)                                                                                         \
  if (deep)                                                                                                    \
    hipLaunchKernelGGL((k_pf_gemm<E, 8>), blocks, dim3(256), 0, s, w, w2, N, K, codes, scales, S, out, bias);  \
  else                                                                                                         \
    hipLaunchKernelGGL((k_pf_gemm<E, 4>), blocks, dim3(256), 0, s, w, w2, N, K, codes, scales, S, out, bias)
  switch (epi) {
    case PF_STORE: MTG_PF_GEMM(PF_STORE); break;
    case PF_RESID: MTG_PF_GEMM(PF_RESID); break;
    case PF_SWIGLU: MTG_PF_GEMM(PF_SWIGLU); break;
    case PF_BIAS: MTG_PF_GEMM(PF_BIAS); break;
    case PF_BIAS_GELU: MTG_PF_GEMM(PF_BIAS_GELU); break;
    case PF_BIAS_SILU: MTG_PF_GEMM(PF_BIAS_SILU); break;
    default: MTG_PF_GEMM(PF_BIAS_RESID); break;
  }
#undef MTG_PF_GEMM
}

void launch_pf_qk_rope(hipStream_t s, const float* qkv, int S, int past0, int n_heads, int n_kv_heads,
                       const float* q_norm, const float* k_norm, float eps, const float* rope, float* q_out,
                       KvLayer kv) {
  hipLaunchKernelGGL(k_pf_qk_rope, dim3((unsigned)S, (unsigned)(n_heads + 2 * n_kv_heads)), dim3(64), 0, s, qkv, S,
                     past0, n_heads, n_kv_heads, q_norm, k_norm, eps, rope, q_out, kv);
}

void launch_pf_attn(hipStream_t s, const float* q, int n_heads, int n_kv_heads, KvLayer kv, int past0, int S,
                    int8_t* ocodes, float* oscales, float* ofl) {
  const int es = kv.f16 ? 2 : 4;
  AttnBlockArgs a{};
  a.q = q;
  a.k = (const uint8_t*)kv.k;
  a.v = (const uint8_t*)kv.v;
  a.head_bytes = (size_t)kv.max_seq * kHeadDim * es;
  a.key_bytes = kHeadDim * es;
  a.q_stride = a.out_stride = n_heads * kHeadDim;
  a.group = n_heads / n_kv_heads;
  a.past = past0;
  a.S = S;
  a.kvlen = past0 + S;
  a.out = ofl;
  a.ocodes = ocodes;
  a.oscales = oscales;
  const dim3 grid((unsigned)(n_heads / 2), (unsigned)((S + 15) / 16));
#define MTG_PF_ATTN(KVH, OUTQ) \
  hipLaunchKernelGGL((k_attn_block<kHeadDim, KVH, true, OUTQ>), grid, dim3(256), AbLds<kHeadDim>::bytes, s, a)
  if (ofl) {
    if (kv.f16) MTG_PF_ATTN(1, false);
    else MTG_PF_ATTN(0, false);
  } else {
    if (kv.f16) MTG_PF_ATTN(1, true);
    else MTG_PF_ATTN(0, true);
  }
#undef MTG_PF_ATTN
}

}  // namespace mtg
