// The attention half of a decoder layer for one token (gfx950),
//   h = x + out_proj(attention(RoPE(qkv_proj(RMSNorm(x))), KV cache)),
// in three launches (benchmark_decode.py:128-303; the host composition of
// moc_amd/inference/decode_model.py is ~35 launches of 2-4 us and two 9 us
// library products):
//
//  decode_qkv_kernel     the norm, the q/k/v projection, RoPE, and the new K
//                        and V straight into the caches.  Bound by W_qkv's
//                        bytes (25 MB at hidden 2048).
//  decode_attn_kernel    one workgroup per head over the cached positions;
//                        scores, softmax and the weighted sum in f32.  Bound
//                        by the latency of one pass over the head's cache.
//  gemv_residual_kernel  out_proj and the residual add.  Bound by W_out's
//                        bytes (8 MB).
//
// Rounding points are those of the stock composition where a value is stored
// in bf16 there (the norm's output, q/k/v, RoPE's output, the attention
// output, out_proj's output, the sum); scores, probabilities and RoPE's
// products, which it rounds to bf16 in between, stay f32 here.
#include <algorithm>

#include "abi.h"
#include "common.h"

namespace moc {
namespace {

constexpr int kAdWaves = 8;             // waves (one unit of rows each) per workgroup
constexpr int kAdThreads = 64 * kAdWaves;
constexpr int kAdMaxHidden = 4096;      // one 16-byte chunk per thread

// RMSNorm of x [hidden] (norm_w null: x as it is) as bf16 in LDS, the whole
// workgroup together: a row's waves share one copy, where a wave that
// normalised x for itself would pull x and the norm weight through L1 for
// every row of the weight.
__device__ __forceinline__ void stage_normed(const uint16_t* __restrict__ x, const uint16_t* __restrict__ norm_w,
                                             float eps, int hidden, uint4* xs, float* red) {
  const int tid = threadIdx.x, nch = hidden / 8;
  uint4 xv = make_uint4(0, 0, 0, 0), nv = make_uint4(0, 0, 0, 0);
  if (tid < nch) {
    xv = reinterpret_cast<const uint4*>(x)[tid];
    if (norm_w != nullptr) nv = reinterpret_cast<const uint4*>(norm_w)[tid];
  }
  if (norm_w != nullptr) {
    const uint32_t a[4] = {xv.x, xv.y, xv.z, xv.w};
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float lo = __uint_as_float(a[j] << 16), hi = __uint_as_float(a[j] & 0xFFFF0000u);
      ss = fmaf(lo, lo, ss);
      ss = fmaf(hi, hi, ss);
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < kAdWaves; ++w) t += red[w];
    xv = rmsnorm8(xv, nv, rsqrtf(t / static_cast<float>(hidden) + eps));
  }
  if (tid < nch) xs[tid] = xv;
  __syncthreads();
}

// Wave w of workgroup b owns rows 2u, 2u + 1 of W_qkv, u = 8 b + w: a RoPE
// pair of one head of q or k, or two neighbouring dimensions of v.  Both rows
// are requested whole before the norm, so the weight's bytes are in flight
// while the workgroup normalises x.
template <int CHN>
__global__ __launch_bounds__(kAdThreads) void decode_qkv_kernel(
    const uint16_t* __restrict__ x, int hidden, const uint16_t* __restrict__ norm_w, float eps,
    const uint16_t* __restrict__ w, int head_dim, const uint16_t* __restrict__ cos, const uint16_t* __restrict__ sin,
    const int64_t* __restrict__ pos_p, int max_seq, uint16_t* __restrict__ q, uint16_t* __restrict__ k_t,
    uint16_t* __restrict__ v) {
  __shared__ uint4 xs[kAdThreads];
  __shared__ float red[kAdWaves];
  const int lane = threadIdx.x & 63;
  const int row = 2 * (static_cast<int>(blockIdx.x) * kAdWaves + (static_cast<int>(threadIdx.x) >> 6));
  const bool live = row < 3 * hidden;
  const int nch = hidden / 8;
  uint4 w0[CHN], w1[CHN];
#pragma unroll
  for (int i = 0; i < CHN; ++i) {
    const int c = lane + 64 * i;
    const uint16_t* p = w + static_cast<int64_t>(live ? row : 0) * hidden + c * 8;
    w0[i] = c < nch ? *reinterpret_cast<const uint4*>(p) : make_uint4(0, 0, 0, 0);
    w1[i] = c < nch ? *reinterpret_cast<const uint4*>(p + hidden) : make_uint4(0, 0, 0, 0);
  }
  const int64_t pos = *pos_p;
  stage_normed(x, norm_w, eps, hidden, xs, red);
  float s0 = 0.f, s1 = 0.f;
#pragma unroll
  for (int i = 0; i < CHN; ++i) {
    const int c = lane + 64 * i;
    const uint4 xv = c < nch ? xs[c] : make_uint4(0, 0, 0, 0);
    s0 = dot8(w0[i], xv, s0);
    s1 = dot8(w1[i], xv, s1);
  }
  s0 = round_bf16(wave_sum(s0));
  s1 = round_bf16(wave_sum(s1));
  if (!live || lane != 0 || pos < 0 || pos >= max_seq) return;
  const int sect = row / hidden, r = row - sect * hidden;
  const int head = r / head_dim, dim = r - head * head_dim;
  float o0 = s0, o1 = s1;
  if (sect < 2) {
    const int64_t e = pos * (head_dim / 2) + dim / 2;
    const float c = bf16_to_f32(cos[e]), s = bf16_to_f32(sin[e]);
    o0 = s0 * c - s1 * s;
    o1 = s0 * s + s1 * c;
  }
  const uint32_t b0 = f32_to_bf16(o0), b1 = f32_to_bf16(o1);
  if (sect == 0) {
    *reinterpret_cast<uint32_t*>(q + r) = b0 | (b1 << 16);
  } else if (sect == 1) {
    uint16_t* d = k_t + static_cast<int64_t>(r) * max_seq + pos;
    d[0] = static_cast<uint16_t>(b0);
    d[max_seq] = static_cast<uint16_t>(b1);
  } else {
    *reinterpret_cast<uint32_t*>(v + (static_cast<int64_t>(head) * max_seq + pos) * head_dim + dim) = b0 | (b1 << 16);
  }
}

// One head per workgroup.  K^T [head_dim, max_seq]: thread (g, j) of 4 x 128
// sums its quarter of the dimensions for positions 2j, 2j + 1 of each block
// of 256; V [max_seq, head_dim]: thread (p, c) of P x head_dim / 8 sums the
// positions p, p + P, ... of its eight dimensions.  The first V rows are
// requested before the scores, so the two passes share one memory latency.
constexpr int kAttnThreads = 512;
constexpr int kAttnVPre = 8;       // V rows per thread requested ahead
constexpr int kAttnMaxSeq = 8192;  // scores held in LDS
constexpr int kAttnMaxDim = 256;

__global__ __launch_bounds__(kAttnThreads) void decode_attn_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_t, const uint16_t* __restrict__ v,
    const int64_t* __restrict__ pos_p, int head_dim, int max_seq, float scale, uint16_t* __restrict__ y) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ float qs[kAttnMaxDim];
  __shared__ float part[4][256];
  __shared__ float wred[2][kAttnThreads / 64];
  float* sc = lds;  // [max_seq rounded to 256], then the V partial sums [P][head_dim]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int head = blockIdx.x;
  const int64_t pos = *pos_p;
  const int n = (pos < 0 || pos >= max_seq) ? 0 : static_cast<int>(pos) + 1;
  const uint16_t* kh = k_t + static_cast<int64_t>(head) * head_dim * max_seq;
  const uint16_t* vh = v + static_cast<int64_t>(head) * max_seq * head_dim;
  const int cpr = head_dim / 8, P = kAttnThreads / cpr;
  const int vp = tid / cpr, vc = tid - vp * cpr;
  uint4 vv[kAttnVPre];
#pragma unroll
  for (int i = 0; i < kAttnVPre; ++i) {
    const int j = vp + P * i;
    vv[i] = vp < P && j < n ? *reinterpret_cast<const uint4*>(vh + static_cast<int64_t>(j) * head_dim + vc * 8)
                            : make_uint4(0, 0, 0, 0);
  }
  if (tid < head_dim) qs[tid] = bf16_to_f32(q[head * head_dim + tid]) * scale;
  __syncthreads();

  // scores of blocks of 256 positions
  const int g = tid >> 7, j2 = (tid & 127) * 2;
  const int d_lo = g * head_dim / 4, d_hi = (g + 1) * head_dim / 4;
  const bool even = (max_seq & 1) == 0;
  float mx = -INFINITY;
  for (int b0 = 0; b0 < n; b0 += 256) {
    const int j = b0 + j2;
    float a0 = 0.f, a1 = 0.f;
    if (j < n) {
      const uint16_t* p = kh + j;
      if (even) {
#pragma unroll 16
        for (int d = d_lo; d < d_hi; ++d) {
          const uint32_t kk = *reinterpret_cast<const uint32_t*>(p + static_cast<int64_t>(d) * max_seq);
          a0 = fmaf(qs[d], __uint_as_float(kk << 16), a0);
          a1 = fmaf(qs[d], __uint_as_float(kk & 0xFFFF0000u), a1);
        }
      } else {
        const int o = j + 1 < n ? 1 : 0;
#pragma unroll 16
        for (int d = d_lo; d < d_hi; ++d) {
          const uint16_t* pd = p + static_cast<int64_t>(d) * max_seq;
          a0 = fmaf(qs[d], bf16_to_f32(pd[0]), a0);
          a1 = fmaf(qs[d], bf16_to_f32(pd[o]), a1);
        }
      }
    }
    part[g][j2] = a0;
    part[g][j2 + 1] = a1;
    __syncthreads();
    if (tid < 256) {
      const float s = (part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]);
      if (b0 + tid < n) {
        sc[b0 + tid] = s;
        mx = fmaxf(mx, s);
      }
    }
    __syncthreads();
  }
  // softmax (f32): NaN scores stay NaN through the sum
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if (lane == 0) wred[0][wave] = mx;
  __syncthreads();
  mx = wred[0][0];
#pragma unroll
  for (int w = 1; w < kAttnThreads / 64; ++w) mx = fmaxf(mx, wred[0][w]);
  float sum = 0.f;
  for (int j = tid; j < n; j += kAttnThreads) {
    const float e = expf(sc[j] - mx);
    sc[j] = e;
    sum += e;
  }
  sum = wave_sum(sum);
  if (lane == 0) wred[1][wave] = sum;
  __syncthreads();
  sum = 0.f;
#pragma unroll
  for (int w = 0; w < kAttnThreads / 64; ++w) sum += wred[1][w];

  // weighted sum of V
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto add = [&](float p, const uint4& t) {
    const uint32_t a[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      acc[2 * e] = fmaf(p, __uint_as_float(a[e] << 16), acc[2 * e]);
      acc[2 * e + 1] = fmaf(p, __uint_as_float(a[e] & 0xFFFF0000u), acc[2 * e + 1]);
    }
  };
  if (vp < P) {
#pragma unroll
    for (int i = 0; i < kAttnVPre; ++i) {
      const int j = vp + P * i;
      if (j < n) add(sc[j], vv[i]);
    }
    for (int j = vp + P * kAttnVPre; j < n; j += P)
      add(sc[j], *reinterpret_cast<const uint4*>(vh + static_cast<int64_t>(j) * head_dim + vc * 8));
  }
  __syncthreads();  // the scores' LDS becomes the partial sums
  if (vp < P) {
#pragma unroll
    for (int e = 0; e < 8; ++e) lds[vp * head_dim + vc * 8 + e] = acc[e];
  }
  __syncthreads();
  if (tid < head_dim) {
    float t = 0.f;
    for (int p = 0; p < P; ++p) t += lds[p * head_dim + tid];
    y[head * head_dim + tid] = f32_to_bf16(t / sum);
  }
}

// y = bf16(res + bf16(W x)): one wave per two rows, x shared in LDS.
template <int CHN>
__global__ __launch_bounds__(kAdThreads) void gemv_residual_kernel(
    const uint16_t* __restrict__ x, int hidden, const uint16_t* __restrict__ w, int rows,
    const uint16_t* __restrict__ res, uint16_t* __restrict__ y) {
  const int lane = threadIdx.x & 63;
  const int row = static_cast<int>(blockIdx.x) * kAdWaves + (static_cast<int>(threadIdx.x) >> 6);
  if (row >= rows) return;
  const int nch = hidden / 8;
  uint4 wv[CHN], xv[CHN];
#pragma unroll
  for (int i = 0; i < CHN; ++i) {
    const int c = lane + 64 * i;
    wv[i] = c < nch ? *reinterpret_cast<const uint4*>(w + static_cast<int64_t>(row) * hidden + c * 8)
                    : make_uint4(0, 0, 0, 0);
    xv[i] = c < nch ? reinterpret_cast<const uint4*>(x)[c] : make_uint4(0, 0, 0, 0);
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < CHN; ++i) s = dot8(wv[i], xv[i], s);
  s = wave_sum(s);
  if (lane == 0) y[row] = f32_to_bf16(bf16_to_f32(res[row]) + round_bf16(s));
}

}  // namespace
}  // namespace moc

using namespace moc;

extern "C" int64_t moc_decode_attention_workspace_size(int64_t hidden) { return hidden > 0 ? 4 * hidden : 0; }

extern "C" int moc_decode_attention_bf16(const void* x, int64_t hidden, int64_t heads, const void* norm_w, float eps,
                                         const void* w_qkv, const void* w_out, const void* cos, const void* sin,
                                         const int64_t* pos, int64_t max_seq, void* k_t, void* v, float scale,
                                         void* y, void* workspace, int64_t workspace_bytes, void* stream) {
  MOC_REQUIRE(heads >= 1 && hidden >= 8 && hidden <= kAdMaxHidden && hidden % heads == 0 && (hidden / heads) % 8 == 0 &&
                  hidden / heads <= kAttnMaxDim,
              "moc_decode_attention_bf16: hidden <= %d in heads of a multiple of 8 up to %d", kAdMaxHidden, kAttnMaxDim);
  MOC_REQUIRE(max_seq >= 1 && max_seq <= kAttnMaxSeq, "moc_decode_attention_bf16: 1 <= max_seq <= %d", kAttnMaxSeq);
  MOC_REQUIRE(eps >= 0.f, "moc_decode_attention_bf16: eps must be >= 0");
  MOC_REQUIRE(x && norm_w && w_qkv && w_out && cos && sin && pos && k_t && v && y && workspace,
              "moc_decode_attention_bf16: null pointer");
  MOC_REQUIRE(aligned16(x) && aligned16(norm_w) && aligned16(w_qkv) && aligned16(w_out) && aligned16(v) &&
                  aligned16(workspace) && reinterpret_cast<uintptr_t>(k_t) % 4 == 0 &&
                  reinterpret_cast<uintptr_t>(y) % 2 == 0,
              "moc_decode_attention_bf16: x, the weights and V must be 16-byte aligned");
  MOC_REQUIRE(workspace_bytes >= moc_decode_attention_workspace_size(hidden),
              "moc_decode_attention_bf16: workspace of %lld bytes required",
              (long long)moc_decode_attention_workspace_size(hidden));
  hipStream_t st = as_stream(stream);
  const int hd = static_cast<int>(hidden), dim = static_cast<int>(hidden / heads), S = static_cast<int>(max_seq);
  uint16_t* q = static_cast<uint16_t*>(workspace);
  uint16_t* o = q + hidden;
  const int chn = (hd / 8 + 63) / 64;
  const dim3 block(kAdThreads), gq(static_cast<unsigned>((3 * hd / 2 + kAdWaves - 1) / kAdWaves)),
      gr(static_cast<unsigned>((hd + kAdWaves - 1) / kAdWaves));
#define MOC_QKV(C)                                                                                                  \
  decode_qkv_kernel<C><<<gq, block, 0, st>>>((const uint16_t*)x, hd, (const uint16_t*)norm_w, eps,                    \
                                             (const uint16_t*)w_qkv, dim, (const uint16_t*)cos, (const uint16_t*)sin, \
                                             pos, S, q, (uint16_t*)k_t, (uint16_t*)v)
  if (chn <= 1) MOC_QKV(1);
  else if (chn <= 2) MOC_QKV(2);
  else if (chn <= 4) MOC_QKV(4);
  else MOC_QKV(8);
#undef MOC_QKV
  int rc = check_launch("decode_qkv_kernel");
  if (rc != MOC_OK) return rc;
  const size_t sc = static_cast<size_t>((S + 255) / 256 * 256) * 4;
  const size_t part = static_cast<size_t>(kAttnThreads / (dim / 8)) * dim * 4;
  decode_attn_kernel<<<dim3(static_cast<unsigned>(heads)), dim3(kAttnThreads), std::max(sc, part), st>>>(
      q, (const uint16_t*)k_t, (const uint16_t*)v, pos, dim, S, scale, o);
  rc = check_launch("decode_attn_kernel");
  if (rc != MOC_OK) return rc;
#define MOC_OUT(C)                                                                                               \
  gemv_residual_kernel<C><<<gr, block, 0, st>>>(o, hd, (const uint16_t*)w_out, hd, (const uint16_t*)x, (uint16_t*)y)
  if (chn <= 1) MOC_OUT(1);
  else if (chn <= 2) MOC_OUT(2);
  else if (chn <= 4) MOC_OUT(4);
  else MOC_OUT(8);
#undef MOC_OUT
  return check_launch("gemv_residual_kernel");
}
