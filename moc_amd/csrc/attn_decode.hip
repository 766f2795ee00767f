// The attention half of a decoder layer for one token (gfx950),
//   h = x + out_proj(attention(RoPE(qkv_proj(RMSNorm(x))), KV cache)),
// in three launches (benchmark_decode.py:128-303; the host composition of
// moc_amd/inference/decode_model.py is ~35 launches of 2-4 us and two 9 us
// library products; the three take 8.2 + 7.5 + 4.2 us at hidden 2048, 16 heads,
// 128 positions, and a 24-layer step went from 3792 to 1331 us with them, then
// to 947 as they and the FFN's kernels were tuned):
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

// One head per workgroup of 16 waves.  The launch is a chain of latencies, so
// everything that does not depend on the scores is requested at once: q, the
// position, the first 256 positions of K^T (which need no position: those past
// it are masked) and of V.
//   K^T [head_dim, max_seq]: thread (g, j) of 8 x 128 sums its eighth of the
//     dimensions (at most DPT) for positions 2j, 2j + 1 of a block of 256;
//   V [max_seq, head_dim]: thread (p, c) of P x head_dim / 8 sums positions p,
//     p + P, ... of its eight dimensions.
// One head of 128 dimensions, 129 positions, in the chain of a decode step:
// 7.4 us (8 waves, four groups of dimensions, the loads behind the position:
// 18.4 us).
constexpr int kAttnThreads = 1024;
constexpr int kAttnWaves = kAttnThreads / 64;
constexpr int kAttnGroups = 8;     // groups of dimensions
constexpr int kAttnVPre = 4;       // V rows per thread requested ahead
constexpr int kAttnMaxSeq = 8192;  // scores held in LDS
constexpr int kAttnMaxDim = 256;

template <int DPT, bool EVEN>
__global__ __launch_bounds__(kAttnThreads) void decode_attn_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_t, const uint16_t* __restrict__ v,
    const int64_t* __restrict__ pos_p, int head_dim, int max_seq, float scale, uint16_t* __restrict__ y) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ float qs[kAttnMaxDim];
  __shared__ float part[kAttnGroups][256];
  __shared__ float wred[2][kAttnWaves];
  float* sc = lds;  // [max_seq rounded to 256], then the V partial sums [P][head_dim]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int head = blockIdx.x;
  const uint16_t* kh = k_t + static_cast<int64_t>(head) * head_dim * max_seq;
  const uint16_t* vh = v + static_cast<int64_t>(head) * max_seq * head_dim;
  const int g = tid >> 7, j2 = (tid & 127) * 2;
  const int dpt = head_dim / kAttnGroups, d0 = g * dpt;
  // two neighbouring positions of one dimension; 0 past the cache
  auto load_k = [&](int d, int j) -> uint32_t {
    const uint16_t* p = kh + static_cast<int64_t>(d0 + d) * max_seq + j;
    if (EVEN) return j < max_seq ? *reinterpret_cast<const uint32_t*>(p) : 0u;
    return j + 1 < max_seq ? p[0] | (static_cast<uint32_t>(p[1]) << 16) : j < max_seq ? p[0] : 0u;
  };
  uint32_t kk[DPT];
#pragma unroll
  for (int d = 0; d < DPT; ++d) kk[d] = d < dpt ? load_k(d, j2) : 0u;
  const int64_t pos = *pos_p;
  if (tid < head_dim) qs[tid] = bf16_to_f32(q[head * head_dim + tid]) * scale;
  const int cpr = head_dim / 8, P = kAttnThreads / cpr;
  const int vp = tid / cpr, vc = tid - vp * cpr;
  uint4 vv[kAttnVPre];
#pragma unroll
  for (int i = 0; i < kAttnVPre; ++i) {
    const int j = vp + P * i;
    vv[i] = vp < P && j < max_seq ? *reinterpret_cast<const uint4*>(vh + static_cast<int64_t>(j) * head_dim + vc * 8)
                                  : make_uint4(0, 0, 0, 0);
  }
  const int n = (pos < 0 || pos >= max_seq) ? 0 : static_cast<int>(pos) + 1;
  __syncthreads();

  // scores of blocks of 256 positions
  float mx = -INFINITY;
  for (int b0 = 0; b0 < n; b0 += 256) {
    if (b0 > 0) {
      __syncthreads();  // the block before is summed
#pragma unroll
      for (int d = 0; d < DPT; ++d) kk[d] = d < dpt ? load_k(d, b0 + j2) : 0u;
    }
    float a0 = 0.f, a1 = 0.f;
#pragma unroll
    for (int d = 0; d < DPT; ++d)
      if (d < dpt) {
        a0 = fmaf(qs[d0 + d], __uint_as_float(kk[d] << 16), a0);
        a1 = fmaf(qs[d0 + d], __uint_as_float(kk[d] & 0xFFFF0000u), a1);
      }
    *reinterpret_cast<float2*>(&part[g][j2]) = make_float2(a0, a1);
    __syncthreads();
    if (tid < 256 && b0 + tid < n) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < kAttnGroups; ++i) s += part[i][tid];
      sc[b0 + tid] = s;
      mx = fmaxf(mx, s);
    }
  }
  // softmax (a NaN score makes the sum NaN)
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if (lane == 0) wred[0][wave] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; ++w) mx = fmaxf(mx, wred[0][w]);  // the waves that hold scores
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
  for (int w = 0; w < kAttnWaves; ++w) sum += wred[1][w];

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
    float4* o = reinterpret_cast<float4*>(lds + vp * head_dim + vc * 8);
    o[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
    o[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
  }
  __syncthreads();
  // thread (s, d) of S x head_dim adds the partial sums s, s + S, ...
  const int S = min(kAttnGroups, kAttnThreads / head_dim), sg = tid / head_dim, sd = tid - sg * head_dim;
  float* fin = &part[0][0];  // S head_dim <= 2048 floats
  if (sg < S) {
    float t = 0.f;
    for (int p = sg; p < P; p += S) t += lds[p * head_dim + sd];
    fin[sg * head_dim + sd] = t;
  }
  __syncthreads();
  if (tid < head_dim) {
    float t = 0.f;
    for (int s = 0; s < S; ++s) t += fin[s * head_dim + tid];
    y[head * head_dim + tid] = f32_to_bf16(t / sum);
  }
}

// y = bf16(res + bf16(W x)): one wave per row, its chunks of the row and of x
// in registers (x comes from L2 for every row but the first of an XCD).  Bound
// by the launch and one round of loads: 4.2 us at 2048 x 2048 (8 MB).
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
  const dim3 ga(static_cast<unsigned>(heads)), ba(kAttnThreads);
#define MOC_ATTN(D, E)                                                                                      \
  decode_attn_kernel<D, E><<<ga, ba, std::max(sc, part), st>>>(q, (const uint16_t*)k_t, (const uint16_t*)v, \
                                                               pos, dim, S, scale, o)
  if (S % 2 == 0) {  // two positions of a dimension in one aligned word
    if (dim <= 64) MOC_ATTN(8, true);
    else if (dim <= 128) MOC_ATTN(16, true);
    else MOC_ATTN(32, true);
  } else {
    if (dim <= 64) MOC_ATTN(8, false);
    else if (dim <= 128) MOC_ATTN(16, false);
    else MOC_ATTN(32, false);
  }
#undef MOC_ATTN
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
