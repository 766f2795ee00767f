// Next-token cross entropy of bf16 logits (gfx950), forward and backward
// (moc/model.py:139-144: logits[:, :-1] against labels[:, 1:], mean over the
// labels that are not ignore_index).
//
// The stock form copies the shifted logits, casts them to f32 under autocast,
// and writes f32 log-probabilities, their gradient, its bf16 cast and the
// gradient of the shift: about ten passes over [tokens, vocab].  Here the
// forward reads the logits once where they are and keeps one f32 per token
// (the log of the sum of exponentials) and, for a backward, their copy (a caller
// may change its logits in place before it; the stock loss keeps its own
// log-probabilities); the backward reads them once and writes the gradient
// once, zeros at the positions without a label included.
// Bound: HBM traffic (4096 x 32000: 262 MB forward, as much again for the copy,
// 524 MB backward): 68 us (3.8 TB/s), 110 with the copy, and 88 us (6.0 TB/s,
// part of the logits still in the last-level cache) there, against 190 + 123 and
// 123 + 161 + 166 us of the stock launches.
#include "abi.h"
#include "common.h"

namespace moc {
namespace {

constexpr int kCeThreads = 512;
constexpr int kCeMaxChunks = 16;  // 16-byte chunks of a row a thread holds in registers

__device__ __forceinline__ float ce_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float ce_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

// Sum or maximum over the workgroup, in wave order.
template <bool MAX>
__device__ __forceinline__ float block_reduce(float v, float* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (MAX) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  } else {
    v = wave_sum(v);
  }
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float t = red[0];
#pragma unroll
  for (int w = 1; w < kCeThreads / 64; ++w) t = MAX ? fmaxf(t, red[w]) : t + red[w];
  return t;
}

// The label of logits row r = b seq + t: labels[b, t + 1]; ignore for the last
// position of a sequence.
__device__ __forceinline__ int64_t label_of(const int64_t* __restrict__ labels, int64_t r, int seq, int64_t ignore) {
  return static_cast<uint32_t>(r) % static_cast<uint32_t>(seq) == static_cast<uint32_t>(seq) - 1 ? ignore : labels[r + 1];
}

// One workgroup per row: the row in registers (NC chunks a thread), its maximum,
// the sum of exponentials; lse[r] and loss[r] (0 where ignored; NaN for a
// label outside the vocabulary, which the stock loss refuses: the loss and that
// row's gradient are then NaN).  keep (may be null): every row's copy.
template <int NC>
__global__ __launch_bounds__(kCeThreads) void ce_forward_kernel(const uint16_t* __restrict__ x, int64_t ld, int vocab,
                                                                int seq, const int64_t* __restrict__ labels,
                                                                int64_t ignore, float* __restrict__ lse,
                                                                float* __restrict__ loss,
                                                                uint16_t* __restrict__ keep, int64_t ldk) {
  __shared__ float red[kCeThreads / 64];
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x;
  const int64_t label = label_of(labels, r, seq, ignore);
  const uint16_t* row = x + r * ld;
  const int n8 = vocab / 8;
  if (label == ignore) {  // uniform over the workgroup
    if (keep != nullptr)
      for (int c = tid; c < n8; c += kCeThreads)
        reinterpret_cast<uint4*>(keep + r * ldk)[c] = reinterpret_cast<const uint4*>(row)[c];
    if (tid == 0) {
      lse[r] = 0.f;
      loss[r] = 0.f;
    }
    return;
  }
  uint4 v[NC];
  // all loads in flight before the first is used (95 -> 70 us at 4096 x 32000):
  // past the end a thread reads the last chunk again, which leaves the maximum
  // and is not summed
#pragma unroll
  for (int i = 0; i < NC; ++i) v[i] = reinterpret_cast<const uint4*>(row)[min(tid + kCeThreads * i, n8 - 1)];
  if (keep != nullptr) {
#pragma unroll
    for (int i = 0; i < NC; ++i)
      if (tid + kCeThreads * i < n8) reinterpret_cast<uint4*>(keep + r * ldk)[tid + kCeThreads * i] = v[i];
  }
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) mx = fmaxf(mx, fmaxf(ce_lo(w[e]), ce_hi(w[e])));
  }
  mx = block_reduce<true>(mx, red);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = tid + kCeThreads * i;
    if (c < n8) {
      const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) sum += expf(ce_lo(w[e]) - mx) + expf(ce_hi(w[e]) - mx);
    }
  }
  sum = block_reduce<false>(sum, red);
  if (tid == 0) {
    const float l = mx + logf(sum);
    const bool known = label >= 0 && label < vocab;
    lse[r] = known ? l : NAN;
    loss[r] = known ? l - bf16_to_f32(row[label]) : NAN;
  }
}

// mean[0] = sum of loss over the rows with a label / their number (NaN if
// none), out = mean in the loss dtype, count[0] = 1 / number.
template <bool OUT_F32>
__global__ __launch_bounds__(1024) void ce_mean_kernel(const float* __restrict__ loss, int64_t rows, int seq,
                                                       const int64_t* __restrict__ labels, int64_t ignore,
                                                       void* __restrict__ out, float* __restrict__ inv) {
  __shared__ double ds[16];
  __shared__ int64_t cs[16];
  double s = 0;
  int64_t c = 0;
  for (int64_t r = threadIdx.x; r < rows; r += 1024) {
    if (label_of(labels, r, seq, ignore) != ignore) {
      s += loss[r];
      ++c;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    s += __shfl_xor(s, o);
    c += __shfl_xor(c, o);
  }
  if ((threadIdx.x & 63) == 0) {
    ds[threadIdx.x >> 6] = s;
    cs[threadIdx.x >> 6] = c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; ++w) {
      s += ds[w];
      c += cs[w];
    }
    const float m = static_cast<float>(s / static_cast<double>(c));
    if (OUT_F32) *static_cast<float*>(out) = m;
    else *static_cast<uint16_t*>(out) = f32_to_bf16(m);
    *inv = static_cast<float>(1.0 / static_cast<double>(c));
  }
}

// dx = (exp(x - lse) - [column = label]) g / count as bf16; zeros in rows
// without a label.
template <bool G_F32>
__global__ __launch_bounds__(kCeThreads) void ce_backward_kernel(const uint16_t* __restrict__ x, int64_t ld, int vocab,
                                                                 int seq, const int64_t* __restrict__ labels,
                                                                 int64_t ignore, const float* __restrict__ lse,
                                                                 const float* __restrict__ inv,
                                                                 const void* __restrict__ g,
                                                                 uint16_t* __restrict__ dx, int64_t ldd) {
  const int64_t r = blockIdx.x;
  const int64_t label = label_of(labels, r, seq, ignore);
  uint4* out = reinterpret_cast<uint4*>(dx + r * ldd);
  const int n8 = vocab / 8;
  if (label == ignore) {
    for (int c = threadIdx.x; c < n8; c += kCeThreads) out[c] = make_uint4(0, 0, 0, 0);
    return;
  }
  const float scale = (G_F32 ? *static_cast<const float*>(g) : bf16_to_f32(*static_cast<const uint16_t*>(g))) * *inv;
  const float l = lse[r];
  const uint4* row = reinterpret_cast<const uint4*>(x + r * ld);
  for (int c = threadIdx.x; c < n8; c += kCeThreads) {
    const uint4 v = row[c];
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    const int64_t at = label - 8 * static_cast<int64_t>(c);  // the label's place in this chunk
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = expf(ce_lo(w[e]) - l) - (at == 2 * e ? 1.f : 0.f);
      const float b = expf(ce_hi(w[e]) - l) - (at == 2 * e + 1 ? 1.f : 0.f);
      o[e] = static_cast<uint32_t>(bf16_rne(a * scale)) | (static_cast<uint32_t>(bf16_rne(b * scale)) << 16);
    }
    out[c] = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

int ce_check(const char* name, const void* x, int64_t ld, int64_t batch, int64_t seq, int64_t vocab,
             const int64_t* labels) {
  MOC_REQUIRE(batch >= 1 && seq >= 1 && batch * seq <= (1LL << 22) && vocab >= 8 && vocab % 8 == 0 &&
                  vocab <= 8LL * kCeThreads * kCeMaxChunks,
              "%s: up to 2^22 positions, vocabulary a multiple of 8 up to %d", name, 8 * kCeThreads * kCeMaxChunks);
  MOC_REQUIRE(x && labels && aligned16(x) && ld % 8 == 0 && ld >= vocab, "%s: logits need 16-byte aligned rows", name);
  return MOC_OK;
}

}  // namespace
}  // namespace moc

using namespace moc;

extern "C" int moc_next_token_loss_forward_keep(const void* logits, int64_t ld, int64_t batch, int64_t seq,
                                                int64_t vocab, const int64_t* labels, int64_t ignore_index, float* lse,
                                                float* row_loss, void* loss, int loss_dtype, float* inv_count,
                                                void* keep, int64_t ldk, void* stream) {
  int rc = ce_check("moc_next_token_loss_forward", logits, ld, batch, seq, vocab, labels);
  if (rc != MOC_OK) return rc;
  MOC_REQUIRE(lse && row_loss && loss && inv_count && (loss_dtype == MOC_BF16 || loss_dtype == MOC_F32),
              "moc_next_token_loss_forward: null output or bad loss dtype");
  MOC_REQUIRE(keep == nullptr || (aligned16(keep) && ldk % 8 == 0 && ldk >= vocab),
              "moc_next_token_loss_forward: the copy needs 16-byte aligned rows");
  hipStream_t st = as_stream(stream);
  const int64_t rows = batch * seq;
  const dim3 grid(static_cast<unsigned>(rows));
  const int nc = static_cast<int>((vocab / 8 + kCeThreads - 1) / kCeThreads);
#define MOC_CE(N)                                                                                             \
  ce_forward_kernel<N><<<grid, kCeThreads, 0, st>>>(static_cast<const uint16_t*>(logits), ld, (int)vocab, (int)seq, \
                                                    labels, ignore_index, lse, row_loss,                       \
                                                    static_cast<uint16_t*>(keep), ldk)
  if (nc <= 2) MOC_CE(2);
  else if (nc <= 4) MOC_CE(4);
  else if (nc <= 8) MOC_CE(8);
  else MOC_CE(16);
#undef MOC_CE
  rc = check_launch("ce_forward_kernel");
  if (rc != MOC_OK) return rc;
  if (loss_dtype == MOC_F32)
    ce_mean_kernel<true><<<1, 1024, 0, st>>>(row_loss, rows, (int)seq, labels, ignore_index, loss, inv_count);
  else
    ce_mean_kernel<false><<<1, 1024, 0, st>>>(row_loss, rows, (int)seq, labels, ignore_index, loss, inv_count);
  return check_launch("ce_mean_kernel");
}

extern "C" int moc_next_token_loss_forward(const void* logits, int64_t ld, int64_t batch, int64_t seq, int64_t vocab,
                                           const int64_t* labels, int64_t ignore_index, float* lse, float* row_loss,
                                           void* loss, int loss_dtype, float* inv_count, void* stream) {
  return moc_next_token_loss_forward_keep(logits, ld, batch, seq, vocab, labels, ignore_index, lse, row_loss, loss,
                                          loss_dtype, inv_count, nullptr, 0, stream);
}

extern "C" int moc_next_token_loss_backward(const void* logits, int64_t ld, int64_t batch, int64_t seq, int64_t vocab,
                                            const int64_t* labels, int64_t ignore_index, const float* lse,
                                            const float* inv_count, const void* grad_loss, int loss_dtype,
                                            void* dlogits, int64_t ldd, void* stream) {
  int rc = ce_check("moc_next_token_loss_backward", logits, ld, batch, seq, vocab, labels);
  if (rc != MOC_OK) return rc;
  MOC_REQUIRE(lse && inv_count && grad_loss && dlogits && aligned16(dlogits) && ldd % 8 == 0 && ldd >= vocab &&
                  (loss_dtype == MOC_BF16 || loss_dtype == MOC_F32),
              "moc_next_token_loss_backward: null or unaligned operand");
  hipStream_t st = as_stream(stream);
  const dim3 grid(static_cast<unsigned>(batch * seq));
  const auto* x = static_cast<const uint16_t*>(logits);
  auto* d = static_cast<uint16_t*>(dlogits);
  if (loss_dtype == MOC_F32)
    ce_backward_kernel<true><<<grid, kCeThreads, 0, st>>>(x, ld, (int)vocab, (int)seq, labels, ignore_index, lse,
                                                          inv_count, grad_loss, d, ldd);
  else
    ce_backward_kernel<false><<<grid, kCeThreads, 0, st>>>(x, ld, (int)vocab, (int)seq, labels, ignore_index, lse,
                                                           inv_count, grad_loss, d, ldd);
  return check_launch("ce_backward_kernel");
}
