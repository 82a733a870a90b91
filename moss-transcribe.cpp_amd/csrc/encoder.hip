// encoder.hip - the Whisper audio encoder and the audio adaptor on the device
// (reference WhisperEncoder::encode, src/whisper_encoder.cpp:103-209, and
// AudioAdaptor::apply, src/audio_adaptor.cpp:38-97).
//
//   conv stem  k_enc_conv_mma: conv1d (kernel 3, pad 1) on f32 MFMA, one fma
//              chain per output over (input channel, tap), + bias, GELU (erf);
//              conv2 (stride 2) also adds the positional embedding and writes
//              [rows][d]
//   layers     k_enc_ln: LayerNorm (mean and variance as double sums over 64
//              lane partials, butterfly) -> q8_0 codes for the next GEMM;
//              q / k / v / out / fc1 / fc2 on the block GEMM of the prefill
//              (q8_0 weights x q8_0 activations, int8 MFMA; q | k | v as one
//              matrix: 1,500 rows 43 -> 32 us) with bias, GELU or
//              residual epilogues; k_attn_block (attn_block.hpp): bidirectional
//              attention on f32 MFMA, 32 query rows of one head per workgroup
//   adaptor    merge consecutive rows (a view), fc1 + SiLU, fc2, LayerNorm
// Every reduction keeps the oracle's order (oracle/oracle.cpp, encoder
// section), so results equal it bit for bit.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "attn_block.hpp"
#include "device_common.hpp"
#include "mtg_internal.hpp"

namespace mtg {
namespace {
using namespace dev;

constexpr int kEncHd = 64;      // head_dim
constexpr int kEncMaxChunks = 32;  // rows <= 2048
constexpr int kConvTile = 64;   // outputs per conv workgroup: 64 rows x 64 channels
constexpr int kConvIcb = 16;    // input channels staged per step

// ------------------------------------------------------------- conv stem ---
// out = gelu(conv(x) + b) (+ pos) on f32 MFMA: the conv as a GEMM over
// n = 3 c + k (input channel c, tap k), out[t][o] = sum_n w[o][n] X[n][t] with
// X[n][t] = x[c][t * STRIDE + k - 1] (0 outside the frames). One MFMA chain per
// 16 x 16 output tile over n in order is the canonical fma chain (tap fastest).
// Workgroup: outputs o0 .. o0 + 63 x t0 .. t0 + 63; wave w: channels
// o0 + 16 w + i (A = w rows) x four 16-row tiles of t (B = X columns). Per block
// of 16 input channels (48 values of n) the w slab (element n = 4 s + g at
// g * 12 + s) and the x rows are staged in LDS; the next block's loads are in
// flight during the current block's MFMAs.
// TRANS: out [OC][OL] (conv2's input layout), else out [OL][OC].
constexpr int kCvNb = 3 * kConvIcb;  // values of n per staged block
constexpr int kCvWs = kCvNb + 4;     // w slab row stride (floats)
template <int STRIDE, bool TRANS>
__global__ void __launch_bounds__(256)
k_enc_conv_mma(const float* __restrict__ w, const float* __restrict__ b, const float* __restrict__ x, int IC, int L,
               int OC, const float* __restrict__ pos, float* __restrict__ out) {
  constexpr int XW = kConvTile * STRIDE + 2;
  constexpr int XN = (kConvIcb * XW + 255) / 256;  // x values per thread and block
  __shared__ __align__(16) float xs[kConvIcb * XW];
  __shared__ __align__(16) float ws[kConvTile * kCvWs];
  const int OL = (L - 1) / STRIDE + 1;
  const int t0 = blockIdx.x * kConvTile, o0 = blockIdx.y * kConvTile;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 15, g = lane >> 4;
  const int p0 = t0 * STRIDE - 1;  // the input position of tap 0 of row t0
  // this lane's x offsets in the staged block: n = 4 s + g -> (c, k) = (n / 3, n % 3)
  int xo[12];
#pragma unroll
  for (int s = 0; s < 12; ++s) {
    const int n = 4 * s + g;
    xo[s] = (n / 3) * XW + n % 3 + j * STRIDE;
  }
  v4f wr[3];
  float xr[XN];
  auto load = [&](int ic0) {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      const int i = tid + 256 * u, o = i / (kCvNb / 4), q = i % (kCvNb / 4);
      wr[u] = *(const v4f*)(w + (size_t)(o0 + o) * IC * 3 + (size_t)ic0 * 3 + 4 * q);
    }
#pragma unroll
    for (int u = 0; u < XN; ++u) {
      const int i = tid + 256 * u, c = i / XW, p = p0 + i % XW;
      xr[u] = (i < kConvIcb * XW && p >= 0 && p < L) ? x[(size_t)(ic0 + min(c, kConvIcb - 1)) * L + min(max(p, 0), L - 1)]
                                                      : 0.0f;
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      const int i = tid + 256 * u, o = i / (kCvNb / 4), q = i % (kCvNb / 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) ws[o * kCvWs + e * 12 + q] = wr[u][e];  // n = 4 q + e
    }
#pragma unroll
    for (int u = 0; u < XN; ++u) {
      const int i = tid + 256 * u;
      if (i < kConvIcb * XW) xs[i] = xr[u];
    }
  };
  v4f acc[4];
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) acc[tt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  load(0);
  for (int ic0 = 0; ic0 < IC; ic0 += kConvIcb) {
    __syncthreads();  // the previous block's operands are consumed
    stage();
    __syncthreads();
    if (ic0 + kConvIcb < IC) load(ic0 + kConvIcb);
    v4f a[3];
    const float* wrow = ws + (16 * wave + j) * kCvWs + g * 12;
#pragma unroll
    for (int u = 0; u < 3; ++u) a[u] = *(const v4f*)(wrow + 4 * u);
#pragma unroll
    for (int s = 0; s < 12; ++s)
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
        acc[tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s >> 2][s & 3], xs[xo[s] + 16 * tt * STRIDE], acc[tt], 0, 0,
                                                       0);
  }
  // acc[tt][r]: output channel o0 + 16 wave + 4 g + r, row t0 + 16 tt + j
  const int ob = o0 + 16 * wave + 4 * g;
  const v4f bias = *(const v4f*)(b + ob);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = __fadd_rn(acc[2 * h + e / 4][e % 4], bias[e % 4]);
    dev_gelu_erf_n<8>(y);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = t0 + 16 * (2 * h + u) + j;
      if (t >= OL) continue;
      v4f v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = y[4 * u + r];
      if (pos) {
        const v4f pv = *(const v4f*)(pos + (size_t)t * OC + ob);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = __fadd_rn(v[r], pv[r]);
      }
      if constexpr (TRANS) {
#pragma unroll
        for (int r = 0; r < 4; ++r) out[(size_t)(ob + r) * OL + t] = v[r];
      } else {
        *(v4f*)(out + (size_t)t * OC + ob) = v;
      }
    }
  }
}

// ------------------------------------------------------------ LayerNorm ----
// One wave per row of 1024 (lane l: elements 16 l .. 16 l + 15): mean and
// variance as double sums of the lanes' sequential partials, wave_sum_d; y =
// ((x - mean) * scale) * w + b with scale = 1 / sqrt(variance + eps). codes /
// scales (nullable): y as q8_0; yout (nullable): y as f32.
__global__ void __launch_bounds__(256)
k_enc_ln(const float* __restrict__ src, int S, const float* __restrict__ w, const float* __restrict__ b, float eps,
         int8_t* __restrict__ codes, float* __restrict__ scales, float* __restrict__ yout) {
  constexpr int D = 1024;
  const int row = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= S) return;
  const float* xr = src + (size_t)row * D + 16 * lane;
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
  for (int e = 0; e < 16; ++e) s = __dadd_rn(s, (double)v[e]);
  s = wave_sum_d(s);
  const float mean = (float)__ddiv_rn(s, (double)D);
  double s2 = 0.0;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    v[e] = __fsub_rn(v[e], mean);
    s2 = __dadd_rn(s2, (double)__fmul_rn(v[e], v[e]));
  }
  s2 = wave_sum_d(s2);
  const float variance = (float)__ddiv_rn(s2, (double)D);
  const float scale = dev_rms_scale(variance, eps);  // 1 / sqrt(variance + eps), correctly rounded
  float y[16];
#pragma unroll
  for (int e = 0; e < 16; ++e)
    y[e] = __fadd_rn(__fmul_rn(__fmul_rn(v[e], scale), w[16 * lane + e]), b[16 * lane + e]);
  if (yout)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *(v4f*)(yout + (size_t)row * D + 16 * lane + 4 * i) = v4f{y[4 * i], y[4 * i + 1], y[4 * i + 2], y[4 * i + 3]};
  if (codes) {
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
      for (int q = 0; q < 4; ++q) u |= (uint32_t)(uint8_t)(int8_t)rintf(__fmul_rn(y[4 * w4 + q], id)) << (8 * q);
      packed[w4] = u;
    }
    *(uint4*)(codes + q8_rows_code(S, row, lane)) = make_uint4(packed[0], packed[1], packed[2], packed[3]);
    if ((lane & 1) == 0) scales[q8_rows_scale(S, row, lane / 2)] = __half2float(__float2half_rn(d));
  }
}

size_t q8_tiles_bytes(int n, int k) { return (size_t)(n / 16) * (k / kPairK) * kUnitBytes; }

}  // namespace
}  // namespace mtg

// ------------------------------------------------------------------ host ---
using namespace mtg;

struct mtg_encoder {
  mtg_encoder_hparams hp{};
  int rows = 0;  // encoder output rows per chunk
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  std::vector<void*> allocs;
  std::string error;
  double last_ms = 0.0;
  int last_rows = 0;
  struct Layer {
    float *attn_ln_w, *attn_ln_b, *qkv_b, *o_b, *ffn_ln_w, *ffn_ln_b, *fc1_b, *fc2_b;
    uint8_t *qkv_w, *o_w, *fc1_w, *fc2_w;  // q | k | v: one matrix of 3 d_model rows
  };
  std::vector<Layer> layers;
  float *conv1_w = nullptr, *conv1_b = nullptr, *conv2_w = nullptr, *conv2_b = nullptr, *pos = nullptr,
        *ln_post_w = nullptr, *ln_post_b = nullptr;
  uint8_t *ad_fc1_w = nullptr, *ad_fc2_w = nullptr;
  float *ad_fc1_b = nullptr, *ad_fc2_b = nullptr, *ad_ln_w = nullptr, *ad_ln_b = nullptr;
  // activations
  float *mel = nullptr, *c1 = nullptr, *x = nullptr, *qkv = nullptr, *a = nullptr,
        *f = nullptr, *out_rows = nullptr, *in_rows = nullptr, *h1 = nullptr, *h2 = nullptr, *ad_out = nullptr;
  int8_t* codes = nullptr;
  float* scales = nullptr;
  // f16 / q4_K matrices (GGUF row layout): the GEMMs' activation (f16 values or
  // q8_K blocks) and the LayerNorm rows it is made from
  int wtype = MTG_TYPE_Q8_0;
  WtAct act{};
  float* xn = nullptr;

  ~mtg_encoder() {
    for (void* p : allocs) (void)hipFree(p);
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (stream) (void)hipStreamDestroy(stream);
  }
  int fail(int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    error = buf;
    return code;
  }
  int check(hipError_t e, const char* what) {
    return e == hipSuccess ? MTG_OK : fail(MTG_ERR_DEVICE, "%s: %s", what, hipGetErrorString(e));
  }
  void* dalloc(size_t bytes) {
    void* p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) return nullptr;
    allocs.push_back(p);
    return p;
  }
  float* up_f(const float* src, size_t n, int& rc) {
    if (rc) return nullptr;
    if (!src) {
      rc = fail(MTG_ERR_INVALID, "a tensor pointer is NULL");
      return nullptr;
    }
    float* d = (float*)dalloc(n * 4);
    if (!d) {
      rc = fail(MTG_ERR_NOMEM, "device memory");
      return nullptr;
    }
    rc = check(hipMemcpy(d, src, n * 4, hipMemcpyHostToDevice), "upload");
    return d;
  }
  uint8_t* up_q8(const void* src, int n, int kk, uint8_t* staging, int& rc, uint8_t* at) {
    if (rc) return nullptr;
    if (!src) {
      rc = fail(MTG_ERR_INVALID, "a tensor pointer is NULL");
      return nullptr;
    }
    uint8_t* d = at ? at : (uint8_t*)dalloc(q8_tiles_bytes(n, kk));
    if (!d) {
      rc = fail(MTG_ERR_NOMEM, "device memory");
      return nullptr;
    }
    const size_t raw = (size_t)n * (kk / 32) * 34;
    if ((rc = check(hipMemcpy(staging, src, raw, hipMemcpyHostToDevice), "upload"))) return nullptr;
    launch_q8_retile(stream, staging, n, kk, d);
    if ((rc = check(hipGetLastError(), "retile"))) return nullptr;
    rc = check(hipStreamSynchronize(stream), "retile");
    return d;
  }
  // bytes of an n x kk matrix on the device
  size_t w_bytes(int n, int kk) const {
    if (wtype == MTG_TYPE_Q8_0) return q8_tiles_bytes(n, kk);
    return (size_t)n * (wtype == MTG_TYPE_F16   ? (size_t)kk * 2
                        : wtype == MTG_TYPE_F32 ? (size_t)kk * 4
                                                : (size_t)(kk / 256) * 144);
  }
  // an n x kk matrix: q8_0 re-tiled for the int8 MFMA GEMM, f16 / f32 / q4_K as they are;
  // into memory of its own, or to `at`
  uint8_t* up_w(const void* src, int n, int kk, uint8_t* staging, int& rc, uint8_t* at = nullptr) {
    if (wtype == MTG_TYPE_Q8_0) return up_q8(src, n, kk, staging, rc, at);
    if (rc) return nullptr;
    if (!src) {
      rc = fail(MTG_ERR_INVALID, "a tensor pointer is NULL");
      return nullptr;
    }
    const size_t bytes = w_bytes(n, kk);
    uint8_t* d = at ? at : (uint8_t*)dalloc(bytes);
    if (!d) {
      rc = fail(MTG_ERR_NOMEM, "device memory");
      return nullptr;
    }
    rc = check(hipMemcpy(d, src, bytes, hipMemcpyHostToDevice), "upload");
    return d;
  }
  // src rows as the next GEMM's activation
  void quant(const float* src, int S, int K) {
    if (wtype == MTG_TYPE_Q8_0) launch_pf_quant(stream, src, S, K, codes, scales);
    else launch_pf_act_wt(stream, wtype, src, S, K, nullptr, 0.0f, act);
  }
  void gemm(int epi, const uint8_t* w, int N, int K, int S, float* out, const float* bias) {
    if (wtype == MTG_TYPE_Q8_0) launch_pf_gemm(stream, epi, w, nullptr, N, K, codes, scales, S, out, bias);
    else launch_pf_gemm_wt(stream, wtype, epi, w, nullptr, N, K, act, S, out, bias);
  }
  // LayerNorm of S rows of d_model: as the next GEMM's activation (q8), or as f32
  // rows in yout
  void ln(const float* src, int S, const float* w, const float* b, float eps, bool q8, float* yout) {
    if (q8 && wtype != MTG_TYPE_Q8_0) {
      hipLaunchKernelGGL(k_enc_ln, dim3((S + 3) / 4), dim3(256), 0, stream, src, S, w, b, eps, nullptr, nullptr, xn);
      quant(xn, S, hp.d_model);
      return;
    }
    hipLaunchKernelGGL(k_enc_ln, dim3((S + 3) / 4), dim3(256), 0, stream, src, S, w, b, eps, q8 ? codes : nullptr,
                       q8 ? scales : nullptr, yout);
  }
};

extern "C" {

int mtg_encoder_create(const mtg_encoder_desc* d, mtg_encoder** out) {
  if (!d || !out) return MTG_ERR_INVALID;
  *out = nullptr;
  const mtg_encoder_hparams& hp = d->hp;
  const int wt = d->weight_type;
  const bool wt_ok = wt == MTG_TYPE_Q8_0 ||
                     ((wt == MTG_TYPE_F16 || wt == MTG_TYPE_F32 || wt == MTG_TYPE_Q4_K) &&
                      pf_gemm_wt_supported(wt, hp.d_model) &&
                      pf_gemm_wt_supported(wt, hp.ffn) && pf_gemm_wt_supported(wt, hp.hidden) &&
                      pf_gemm_wt_supported(wt, hp.d_model * hp.merge));
  if (!wt_ok || hp.d_model != 1024 || hp.hidden != 1024 || hp.n_heads <= 0 ||
      hp.d_model / hp.n_heads != kEncHd || hp.d_model % hp.n_heads || hp.ffn % 64 || hp.n_mels % kConvIcb ||
      hp.n_mels <= 0 || hp.merge <= 0 || hp.n_layers < 0 || hp.n_frames < 2 ||
      (hp.n_frames - 1) / 2 + 1 > 64 * kEncMaxChunks)
    return MTG_ERR_UNSUPPORTED;
  if (!d->layers && hp.n_layers > 0) return MTG_ERR_INVALID;
  mtg_encoder* e = new (std::nothrow) mtg_encoder();
  if (!e) return MTG_ERR_NOMEM;
  e->hp = hp;
  e->wtype = wt;
  const int D = hp.d_model, F = hp.ffn, M = hp.n_mels, NF = hp.n_frames, R = (NF - 1) / 2 + 1, H = hp.hidden,
            IN = D * hp.merge;
  e->rows = R;
  int rc = e->check(hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking), "stream");
  if (!rc) rc = e->check(hipEventCreate(&e->ev0), "event");
  if (!rc) rc = e->check(hipEventCreate(&e->ev1), "event");
  if (!rc) rc = e->check(prepare_kernels_pf_wt(), "kernel attributes");
  // staging for the raw q8_0 rows of the largest matrix
  size_t raw_max = (size_t)std::max(F, std::max(D, H)) * (std::max(F, IN) / 32) * 34;
  uint8_t* staging = rc ? nullptr : (uint8_t*)e->dalloc(raw_max);
  if (!rc && !staging) rc = e->fail(MTG_ERR_NOMEM, "device memory");
  e->conv1_w = e->up_f(d->conv1_w, (size_t)D * M * 3, rc);
  e->conv1_b = e->up_f(d->conv1_b, D, rc);
  e->conv2_w = e->up_f(d->conv2_w, (size_t)D * D * 3, rc);
  e->conv2_b = e->up_f(d->conv2_b, D, rc);
  e->pos = e->up_f(d->pos_embd, (size_t)R * D, rc);
  e->ln_post_w = e->up_f(d->ln_post_w, D, rc);
  e->ln_post_b = e->up_f(d->ln_post_b, D, rc);
  std::vector<float> qkv_b((size_t)3 * D, 0.0f);
  for (int l = 0; l < hp.n_layers && !rc; ++l) {
    const mtg_encoder_layer& s = d->layers[l];
    mtg_encoder::Layer L{};
    L.attn_ln_w = e->up_f(s.attn_ln_w, D, rc);
    L.attn_ln_b = e->up_f(s.attn_ln_b, D, rc);
    const size_t part = e->w_bytes(D, D);
    L.qkv_w = rc ? nullptr : (uint8_t*)e->dalloc(3 * part);
    if (!rc && !L.qkv_w) rc = e->fail(MTG_ERR_NOMEM, "device memory");
    e->up_w(s.q_w, D, D, staging, rc, L.qkv_w);
    e->up_w(s.k_w, D, D, staging, rc, L.qkv_w + part);
    e->up_w(s.v_w, D, D, staging, rc, L.qkv_w + 2 * part);
    L.o_w = e->up_w(s.o_w, D, D, staging, rc);
    // k has no bias: + 0 leaves its sums as they are (their chains start at +0, so none is
    // -0 unless every f32 product of one underflows)
    if (!rc && (!s.q_b || !s.v_b)) rc = e->fail(MTG_ERR_INVALID, "a tensor pointer is NULL");
    if (!rc) {
      std::copy(s.q_b, s.q_b + D, qkv_b.begin());
      std::copy(s.v_b, s.v_b + D, qkv_b.begin() + 2 * D);
    }
    L.qkv_b = e->up_f(qkv_b.data(), 3 * (size_t)D, rc);
    L.o_b = e->up_f(s.o_b, D, rc);
    L.ffn_ln_w = e->up_f(s.ffn_ln_w, D, rc);
    L.ffn_ln_b = e->up_f(s.ffn_ln_b, D, rc);
    L.fc1_w = e->up_w(s.fc1_w, F, D, staging, rc);
    L.fc1_b = e->up_f(s.fc1_b, F, rc);
    L.fc2_w = e->up_w(s.fc2_w, D, F, staging, rc);
    L.fc2_b = e->up_f(s.fc2_b, D, rc);
    e->layers.push_back(L);
  }
  e->ad_fc1_w = e->up_w(d->ad_fc1_w, H, IN, staging, rc);
  e->ad_fc1_b = e->up_f(d->ad_fc1_b, H, rc);
  e->ad_fc2_w = e->up_w(d->ad_fc2_w, H, H, staging, rc);
  e->ad_fc2_b = e->up_f(d->ad_fc2_b, H, rc);
  e->ad_ln_w = e->up_f(d->ad_ln_w, H, rc);
  e->ad_ln_b = e->up_f(d->ad_ln_b, H, rc);
  if (!rc) {
    const size_t RD = (size_t)R * D;
    e->mel = (float*)e->dalloc((size_t)M * NF * 4);
    e->c1 = (float*)e->dalloc((size_t)D * NF * 4);
    e->x = (float*)e->dalloc(RD * 4);
    e->qkv = (float*)e->dalloc(3 * RD * 4);
    e->a = (float*)e->dalloc(RD * 4);
    e->f = (float*)e->dalloc((size_t)R * F * 4);
    e->out_rows = (float*)e->dalloc(RD * 4);
    e->in_rows = (float*)e->dalloc(RD * 4);
    const int N = R / hp.merge + 1;
    e->h1 = (float*)e->dalloc((size_t)N * H * 4);
    e->h2 = (float*)e->dalloc((size_t)N * H * 4);
    e->ad_out = (float*)e->dalloc((size_t)N * H * 4);
    // whole 64-row blocks (q8_rows_code)
    const size_t KC = std::max((size_t)((R + 63) / 64 * 64) * std::max(F, D), (size_t)((N + 63) / 64 * 64) * IN);
    e->codes = (int8_t*)e->dalloc(KC);
    e->scales = (float*)e->dalloc(KC / 32 * 4);
    if (wt == MTG_TYPE_F16) {
      e->act.f16h = (uint16_t*)e->dalloc(KC * 2);
      if (!e->act.f16h) rc = e->fail(MTG_ERR_NOMEM, "device memory");
    } else if (wt == MTG_TYPE_F32) {
      e->act.f32 = (float*)e->dalloc(KC * 4);
      if (!e->act.f32) rc = e->fail(MTG_ERR_NOMEM, "device memory");
    } else if (wt == MTG_TYPE_Q4_K) {
      e->act.q8k.qs = (int8_t*)e->dalloc(KC);
      e->act.q8k.d = (float*)e->dalloc(KC / 256 * 4);
      e->act.q8k.bsums = (int32_t*)e->dalloc(KC / 16 * 4);
      if (!e->act.q8k.qs || !e->act.q8k.d || !e->act.q8k.bsums) rc = e->fail(MTG_ERR_NOMEM, "device memory");
    }
    if (wt != MTG_TYPE_Q8_0) {
      e->xn = (float*)e->dalloc(RD * 4);
      if (!e->xn) rc = e->fail(MTG_ERR_NOMEM, "device memory");
    }
    if (!e->mel || !e->c1 || !e->x || !e->qkv || !e->a || !e->f || !e->out_rows || !e->in_rows ||
        !e->h1 || !e->h2 || !e->ad_out || !e->codes || !e->scales)
      rc = e->fail(MTG_ERR_NOMEM, "device memory");
  }
  if (rc) {
    delete e;
    return rc;
  }
  *out = e;
  return MTG_OK;
}

void mtg_encoder_destroy(mtg_encoder* e) { delete e; }

const char* mtg_encoder_error(const mtg_encoder* e) { return e ? e->error.c_str() : "no encoder"; }

double mtg_encoder_last_ms(const mtg_encoder* e) { return e ? e->last_ms : 0.0; }

int mtg_encoder_encode(mtg_encoder* e, const float* mel, float* out, int32_t* rows_out) {
  if (!e || !mel) return MTG_ERR_INVALID;
  const mtg_encoder_hparams& hp = e->hp;
  const int D = hp.d_model, F = hp.ffn, M = hp.n_mels, NF = hp.n_frames, R = e->rows;
  hipStream_t s = e->stream;
  int rc = e->check(hipMemcpyAsync(e->mel, mel, (size_t)M * NF * 4, hipMemcpyHostToDevice, s), "mel");
  if (rc) return rc;
  if ((rc = e->check(hipEventRecord(e->ev0, s), "event"))) return rc;
  // conv stem
  hipLaunchKernelGGL((k_enc_conv_mma<1, true>), dim3((NF + kConvTile - 1) / kConvTile, D / kConvTile), dim3(256), 0, s,
                     e->conv1_w, e->conv1_b, e->mel, M, NF, D, (const float*)nullptr, e->c1);
  hipLaunchKernelGGL((k_enc_conv_mma<2, false>), dim3((R + kConvTile - 1) / kConvTile, D / kConvTile), dim3(256), 0, s,
                     e->conv2_w, e->conv2_b, e->c1, D, NF, D, e->pos, e->x);
  const dim3 agrid((unsigned)hp.n_heads, (unsigned)((R + 31) / 32));
  AttnBlockArgs attn{};
  attn.q = e->qkv;
  attn.k = (const uint8_t*)(e->qkv + D);
  attn.v = (const uint8_t*)(e->qkv + 2 * D);
  attn.head_bytes = kEncHd * 4;
  attn.key_bytes = 3 * D * 4;
  attn.q_stride = 3 * D;
  attn.out_stride = D;
  attn.S = attn.kvlen = R;
  attn.out = e->a;
  for (const mtg_encoder::Layer& L : e->layers) {
    e->ln(e->x, R, L.attn_ln_w, L.attn_ln_b, 1e-5f, true, nullptr);
    e->gemm(PF_EPI_BIAS, L.qkv_w, 3 * D, D, R, e->qkv, L.qkv_b);
    hipLaunchKernelGGL((k_attn_block<kEncHd, 0, false, false>), agrid, dim3(256), AbLds<kEncHd>::bytes, s, attn);
    e->quant(e->a, R, D);
    e->gemm(PF_EPI_BIAS_RESID, L.o_w, D, D, R, e->x, L.o_b);
    e->ln(e->x, R, L.ffn_ln_w, L.ffn_ln_b, 1e-5f, true, nullptr);
    e->gemm(PF_EPI_BIAS_GELU, L.fc1_w, F, D, R, e->f, L.fc1_b);
    e->quant(e->f, R, F);
    e->gemm(PF_EPI_BIAS_RESID, L.fc2_w, D, F, R, e->x, L.fc2_b);
  }
  e->ln(e->x, R, e->ln_post_w, e->ln_post_b, 1e-5f, false, e->out_rows);
  if ((rc = e->check(hipGetLastError(), "encoder launch"))) return rc;
  if ((rc = e->check(hipEventRecord(e->ev1, s), "event"))) return rc;
  if (out && (rc = e->check(hipMemcpyAsync(out, e->out_rows, (size_t)R * D * 4, hipMemcpyDeviceToHost, s), "rows")))
    return rc;
  if ((rc = e->check(hipStreamSynchronize(s), "encode"))) return rc;
  float ms = 0.0f;
  if ((rc = e->check(hipEventElapsedTime(&ms, e->ev0, e->ev1), "timing"))) return rc;
  e->last_ms = ms;
  e->last_rows = R;
  if (rows_out) *rows_out = R;
  return MTG_OK;
}

int mtg_encoder_adapt(mtg_encoder* e, const float* rows, int32_t T, float* out, int32_t* n_out) {
  if (!e || !out || T < 0) return MTG_ERR_INVALID;
  const mtg_encoder_hparams& hp = e->hp;
  const int D = hp.d_model, H = hp.hidden, IN = D * hp.merge, N = T / hp.merge;
  if (T > e->rows || (!rows && T > e->last_rows))
    return e->fail(MTG_ERR_INVALID, "adapt: %d rows, the encoder holds %d", T, rows ? e->rows : e->last_rows);
  if (n_out) *n_out = N;
  if (N <= 0) return MTG_OK;
  hipStream_t s = e->stream;
  int rc = MTG_OK;
  const float* src = e->out_rows;
  if (rows) {
    if ((rc = e->check(hipMemcpyAsync(e->in_rows, rows, (size_t)N * IN * 4, hipMemcpyHostToDevice, s), "rows")))
      return rc;
    src = e->in_rows;
  }
  if ((rc = e->check(hipEventRecord(e->ev0, s), "event"))) return rc;
  // [D * merge, N]: merge consecutive rows per adaptor row (a plain view)
  e->quant(src, N, IN);
  e->gemm(PF_EPI_BIAS_SILU, e->ad_fc1_w, H, IN, N, e->h1, e->ad_fc1_b);
  e->quant(e->h1, N, H);
  e->gemm(PF_EPI_BIAS, e->ad_fc2_w, H, H, N, e->h2, e->ad_fc2_b);
  e->ln(e->h2, N, e->ad_ln_w, e->ad_ln_b, hp.adaptor_eps, false, e->ad_out);
  if ((rc = e->check(hipGetLastError(), "adaptor launch"))) return rc;
  if ((rc = e->check(hipEventRecord(e->ev1, s), "event"))) return rc;
  if ((rc = e->check(hipMemcpyAsync(out, e->ad_out, (size_t)N * H * 4, hipMemcpyDeviceToHost, s), "adaptor rows")))
    return rc;
  if ((rc = e->check(hipStreamSynchronize(s), "adapt"))) return rc;
  float ms = 0.0f;
  if ((rc = e->check(hipEventElapsedTime(&ms, e->ev0, e->ev1), "timing"))) return rc;
  e->last_ms = ms;
  return MTG_OK;
}

}  // extern "C"
