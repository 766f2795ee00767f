// Causal attention of a decoder block on the matrix cores (gfx950), forward
// and backward, with RoPE applied to q and k as they are read
// (moc/model.py:31-64: qkv_proj's output, rotate the pairs (2i, 2i + 1) of q
// and k, scaled dot products under a causal mask).
//
//   q, k, v: the sections of qkv [batch seq, 3 heads HD]; o [batch seq, heads
//   HD]; lse [batch, heads, seq] = log2 of each query's sum of exp2 scores.
//
// The stock form rotates with nine elementwise launches over copies of q and
// k, and its backward with about thirty more; here q/k/v are read where the
// projection left them and the gradients are written where its backward reads
// them.  Bound: HBM traffic (qkv, o and their gradients once per pass) and the
// latency of a workgroup's few tiles; the products are 5 % of the MFMA rate.
//
// Orientation.  v_mfma_f32_32x32x16 leaves a lane with one column (l & 31) and
// the rows 8 (r >> 2) + 4 (l >> 5) + (r & 3).  Each wave owns 32 columns (its
// queries in the forward and in dQ, its keys in dK/dV), so every softmax
// factor is a per-lane value, and the 16 rows a lane holds are, taken eight at
// a time, a B operand of the next product with its k index permuted to
// {4 h, .., 4 h + 3, 8 + 4 h, ..}, h = l >> 5.  The other operand of that
// product is read from LDS transposed (ds_read_b64_tr_b16) under the same
// permutation, so neither P nor dS ever passes through LDS.
//
// LDS tiles hold 64 rows of HD values; 16-byte chunk c of row r sits in slot
// c ^ f(r), which serves the row-wise b128 reads and the transposing ones.
#include "abi.h"
#include "common.h"

namespace moc {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) i16x4_t lds_i16x4_t;

constexpr int kAtThreads = 256;  // four waves of 32 columns
constexpr int kAtCols = 128;     // columns (queries or keys) per workgroup
constexpr int kAtTile = 64;      // rows per LDS tile of the backward

struct AttnArgs {
  const uint16_t* qkv;
  int64_t ld;         // elements between tokens of qkv (and of dqkv)
  int heads, seq;
  const void *cos, *sin;  // [>= seq, HD / 2]
  float c2;               // scale log2(e)
  float scale;
  uint16_t* o;         // [batch seq, heads HD]
  float* lse;          // [batch, heads, seq]
  const uint16_t* go;  // gradient of o
  float* delta;        // [batch, heads, seq]: sum of go o
  uint16_t* dqkv;
};

__device__ __forceinline__ uint32_t pk(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((cvt_f32x2_t){lo, hi}, cvt_bf16x2_t));
}
__device__ __forceinline__ float lo_f(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi_f(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

// cos and sin of the four pairs of the 8-value chunk c at position pos
template <int HD, bool TF32>
__device__ __forceinline__ void load_angles(const AttnArgs& a, int pos, int c, float (&cs)[4], float (&sn)[4]) {
  const int64_t e = static_cast<int64_t>(pos) * (HD / 2) + 4 * c;
  if (TF32) {
    const float4 x = *reinterpret_cast<const float4*>(static_cast<const float*>(a.cos) + e);
    const float4 y = *reinterpret_cast<const float4*>(static_cast<const float*>(a.sin) + e);
    cs[0] = x.x; cs[1] = x.y; cs[2] = x.z; cs[3] = x.w;
    sn[0] = y.x; sn[1] = y.y; sn[2] = y.z; sn[3] = y.w;
  } else {
    const uint2 x = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(a.cos) + e);
    const uint2 y = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(a.sin) + e);
    cs[0] = lo_f(x.x); cs[1] = hi_f(x.x); cs[2] = lo_f(x.y); cs[3] = hi_f(x.y);
    sn[0] = lo_f(y.x); sn[1] = hi_f(y.x); sn[2] = lo_f(y.y); sn[3] = hi_f(y.y);
  }
}

// The rotation of four pairs with the stock form's rounding points: bf16 tables
// round each product and the sum (bf16 tensor operations); f32 tables promote
// q and k to f32, cast once at the attention.
template <bool TF32>
__device__ __forceinline__ uint4 rotate8(uint4 v, const float (&cs)[4], const float (&sn)[4]) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = lo_f(w[i]), b = hi_f(w[i]);
    if (TF32) {
      o[i] = pk(a * cs[i] - b * sn[i], a * sn[i] + b * cs[i]);
    } else {
      const uint32_t p = pk(a * cs[i], b * sn[i]), q = pk(a * sn[i], b * cs[i]);
      o[i] = pk(lo_f(p) - hi_f(p), lo_f(q) + hi_f(q));
    }
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

template <int HD>
__device__ __forceinline__ int swz(int r) {
  return HD == 64 ? ((r & 7) ^ ((r >> 3) & 1)) : (r & 15);
}

// A ROWS x HD tile on its way to LDS: thread t holds chunks t, t + 256, ...
// (row chunk / (HD / 8)); rows past the sequence are zero.
template <int HD, bool ROT, bool TF32, int ROWS = kAtTile>
struct Tile {
  static constexpr int kN = ROWS * HD / 8 / kAtThreads;
  uint4 v[kN];
  float cs[ROT ? kN : 1][4], sn[ROT ? kN : 1][4];

  __device__ __forceinline__ void load(const AttnArgs& a, const uint16_t* p, int64_t ld, int row0, int tid) {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const int q = tid + kAtThreads * i, r = row0 + q / (HD / 8), c = q % (HD / 8);
      v[i] = r < a.seq ? *reinterpret_cast<const uint4*>(p + r * ld + 8 * c) : make_uint4(0, 0, 0, 0);
      if (ROT) load_angles<HD, TF32>(a, min(r, a.seq - 1), c, cs[i], sn[i]);
    }
  }
  __device__ __forceinline__ void store(char* lds, int tid) const {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const int q = tid + kAtThreads * i, r = q / (HD / 8), c = q % (HD / 8);
      uint4 t = v[i];
      if constexpr (ROT) t = rotate8<TF32>(t, cs[i], sn[i]);
      *reinterpret_cast<uint4*>(lds + r * (HD * 2) + 16 * (c ^ swz<HD>(r))) = t;
    }
  }
};

// Operand of rows blk + (l & 31), values 16 ks + 8 (l >> 5) .. + 7.
template <int HD>
__device__ __forceinline__ bf16x8_t read_rows(const char* lds, int blk, int ks, int lane) {
  const int r = blk + (lane & 31), c = 2 * ks + (lane >> 5);
  return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(lds + r * (HD * 2) + 16 * (c ^ swz<HD>(r))));
}

// Operand of columns col + (l & 31) of the tile, k the rows row + {4 h ..
// 4 h + 3, 8 + 4 h ..} (h = l >> 5): two transposing reads.
template <int HD>
__device__ __forceinline__ bf16x8_t read_cols(const char* lds, int col, int row, int lane) {
  const int i = lane & 15, g = lane >> 4;
  const int r = row + 4 * (g >> 1) + (i >> 2), m = col + 16 * (g & 1) + 4 * (i & 3);
  const char* lo = lds + r * (HD * 2) + 16 * ((m >> 3) ^ swz<HD>(r)) + 8 * (i & 1);
  const char* hi = lds + (r + 8) * (HD * 2) + 16 * ((m >> 3) ^ swz<HD>(r + 8)) + 8 * (i & 1);
  const i16x4_t v[2] = {__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)lo),
                        __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)hi)};
  return __builtin_bit_cast(bf16x8_t, v);
}

// The wave's own 32 columns as a B operand, from memory: values 16 ks +
// 8 (l >> 5) .. + 7 of row r (zero past the sequence).
template <int HD, bool ROT, bool TF32>
__device__ __forceinline__ void load_own(const AttnArgs& a, const uint16_t* p, int64_t ld, int r, int lane,
                                         bf16x8_t (&f)[HD / 16]) {
#pragma unroll
  for (int ks = 0; ks < HD / 16; ++ks) {
    const int c = 2 * ks + (lane >> 5);
    uint4 v = r < a.seq ? *reinterpret_cast<const uint4*>(p + r * ld + 8 * c) : make_uint4(0, 0, 0, 0);
    if constexpr (ROT) {
      float cs[4], sn[4];
      load_angles<HD, TF32>(a, min(r, a.seq - 1), c, cs, sn);
      v = rotate8<TF32>(v, cs, sn);
    }
    f[ks] = __builtin_bit_cast(bf16x8_t, v);
  }
}

__device__ __forceinline__ bf16x8_t pack8(const float* p) {
  const uint32_t w[4] = {pk(p[0], p[1]), pk(p[2], p[3]), pk(p[4], p[5]), pk(p[6], p[7])};
  return __builtin_bit_cast(bf16x8_t, w);
}

__device__ __forceinline__ void zero(f32x16_t& a) {
#pragma unroll
  for (int r = 0; r < 16; ++r) a[r] = 0.f;
}

// Column r's HD values (accumulators [HD / 32], times f) to dst as bf16, for
// ROT rotated back by the position's angles.
template <int HD, bool ROT, bool TF32>
__device__ __forceinline__ void store_own(const AttnArgs& a, const f32x16_t (&acc)[HD / 32], float f, uint16_t* dst,
                                          int pos, int lane) {
#pragma unroll
  for (int b = 0; b < HD / 32; ++b)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int dim = 32 * b + 8 * q + 4 * (lane >> 5);
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = acc[b][4 * q + e] * f;
      if constexpr (ROT) {
        const int64_t e0 = static_cast<int64_t>(pos) * (HD / 2) + dim / 2;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float cs = TF32 ? static_cast<const float*>(a.cos)[e0 + e]
                                : bf16_to_f32(static_cast<const uint16_t*>(a.cos)[e0 + e]);
          const float sn = TF32 ? static_cast<const float*>(a.sin)[e0 + e]
                                : bf16_to_f32(static_cast<const uint16_t*>(a.sin)[e0 + e]);
          const float x = v[2 * e], y = v[2 * e + 1];
          v[2 * e] = x * cs + y * sn;
          v[2 * e + 1] = y * cs - x * sn;
        }
      }
      *reinterpret_cast<uint2*>(dst + dim) = make_uint2(pk(v[0], v[1]), pk(v[2], v[3]));
    }
}

// ------------------------------------------------------------------ forward
// Key tiles of T rows.  P is rounded to bf16 relative to the running maximum,
// which moves once a tile; with T as launch_fwd chooses it, it moves where it
// does in the library attention that the stock composition calls, and the
// outputs agree to the bit on all but at most 2 in 1000 values (36 lengths of 2 to
// 2048 positions, heads of 64 and 128; bf16 tables 4 in 100000 at most, but for
// 17 positions).  With another T 5 to 20 % of them differ by a rounding, which a
// MoC selection after it amplifies.
template <int HD, bool TF32, int T>
__global__ __launch_bounds__(kAtThreads, HD == 64 ? 2 : 1) void attn_fwd_kernel(AttnArgs a) {
  constexpr int KB = T / 32;
  __shared__ __attribute__((aligned(1024))) char lk[T * HD * 2];
  __shared__ __attribute__((aligned(1024))) char lv[T * HD * 2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int head = blockIdx.y, b = blockIdx.z, d = a.heads * HD;
  // the longest rows of the triangle first
  const int col0 = (static_cast<int>(gridDim.x) - 1 - static_cast<int>(blockIdx.x)) * kAtCols;
  const int q0 = col0 + 32 * wave, q = q0 + (lane & 31);
  const uint16_t* base = a.qkv + static_cast<int64_t>(b) * a.seq * a.ld + head * HD;
  bf16x8_t fq[HD / 16];
  load_own<HD, true, TF32>(a, base, a.ld, q, lane, fq);
  f32x16_t acc[HD / 32];
#pragma unroll
  for (int i = 0; i < HD / 32; ++i) zero(acc[i]);
  float m = -INFINITY, l = 0.f;
  const int nt = (min(col0 + kAtCols, a.seq) + T - 1) / T;
  // T = 64: the next tile is requested while this one is multiplied; T = 128
  // has no registers for that at two workgroups a CU, which hide the latency
  // instead
  constexpr bool kAhead = T == 64;
  Tile<HD, true, TF32, T> tk;
  Tile<HD, false, TF32, T> tv;
  if (kAhead) {
    tk.load(a, base + d, a.ld, 0, tid);
    tv.load(a, base + 2 * d, a.ld, 0, tid);
  }
  for (int t = 0; t < nt; ++t) {
    if (!kAhead) {
      tk.load(a, base + d, a.ld, t * T, tid);
      tv.load(a, base + 2 * d, a.ld, t * T, tid);
    }
    tk.store(lk, tid);
    tv.store(lv, tid);
    __syncthreads();
    if (kAhead && t + 1 < nt) {
      tk.load(a, base + d, a.ld, (t + 1) * T, tid);
      tv.load(a, base + 2 * d, a.ld, (t + 1) * T, tid);
    }
    const int k0 = t * T;
    if (k0 <= q0 + 31 && q0 < a.seq) {  // wave-uniform: some key of the tile is visible
      f32x16_t s[KB];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        zero(s[kb]);
#pragma unroll
        for (int ks = 0; ks < HD / 16; ++ks)
          s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_rows<HD>(lk, 32 * kb, ks, lane), fq[ks], s[kb], 0, 0, 0);
      }
      float mx = -INFINITY;
      const bool diag = k0 + T - 1 > q0;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = k0 + 32 * kb + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          float x = s[kb][r] * a.c2;
          if (diag && key > q) x = -INFINITY;
          s[kb][r] = x;
          mx = fmaxf(mx, x);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      // a column with no visible key yet keeps the maximum of 0 for its
      // exponents: every exp2 below is then exp2(-inf) = 0
      const float mn = fmaxf(m, mx), ref = mn == -INFINITY ? 0.f : mn;
      const float alpha = exp2f(m - ref);
      m = mn;
      float sum = 0.f;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = exp2f(s[kb][r] - ref);
          s[kb][r] = p;
          sum += p;
        }
      l = l * alpha + sum;
#pragma unroll
      for (int i = 0; i < HD / 32; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] *= alpha;
#pragma unroll
      for (int st = 0; st < 2 * KB; ++st) {
        float pv[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) pv[e] = s[st >> 1][8 * (st & 1) + e];
        const bf16x8_t fp = pack8(pv);
#pragma unroll
        for (int i = 0; i < HD / 32; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_cols<HD>(lv, 32 * i, 16 * st, lane), fp, acc[i], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  if (q >= a.seq) return;
  l += __shfl_xor(l, 32);
  const int64_t row = static_cast<int64_t>(b) * a.seq + q;
  store_own<HD, false, TF32>(a, acc, 1.0f / l, a.o + row * d + head * HD, 0, lane);
  if (lane < 32) a.lse[(static_cast<int64_t>(b) * a.heads + head) * a.seq + q] = m + log2f(l);
}

// ----------------------------------------------------------------- backward
// dQ: the wave's queries against every key tile they see; also delta.  A
// kernel of its own for each side, recomputing the scores, keeps every sum
// inside one wave: no atomics and no cross-workgroup partials.  Bound by the
// latency of a workgroup's two to four tiles.  4096 tokens of 256, 16 heads of
// 64: dQ 28 us, dK/dV 44 us, forward 20 us; the library's backward is 104 us,
// its forward 50, the RoPE launches around them not counted.
template <int HD, bool TF32>
__global__ __launch_bounds__(kAtThreads) void attn_bwd_q_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(1024))) char lk[kAtTile * HD * 2];
  __shared__ __attribute__((aligned(1024))) char lv[kAtTile * HD * 2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int head = blockIdx.y, b = blockIdx.z, d = a.heads * HD;
  const int col0 = (static_cast<int>(gridDim.x) - 1 - static_cast<int>(blockIdx.x)) * kAtCols;
  const int q0 = col0 + 32 * wave, q = q0 + (lane & 31);
  const int64_t tok0 = static_cast<int64_t>(b) * a.seq;
  const uint16_t* base = a.qkv + tok0 * a.ld + head * HD;
  bf16x8_t fq[HD / 16], fg[HD / 16];
  load_own<HD, true, TF32>(a, base, a.ld, q, lane, fq);
  load_own<HD, false, TF32>(a, a.go + tok0 * d + head * HD, d, q, lane, fg);
  const int64_t st_row = (static_cast<int64_t>(b) * a.heads + head) * a.seq + q;
  float dl = 0.f;
  {
    bf16x8_t fo[HD / 16];
    load_own<HD, false, TF32>(a, a.o + tok0 * d + head * HD, d, q, lane, fo);
#pragma unroll
    for (int ks = 0; ks < HD / 16; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) dl = fmaf(static_cast<float>(fo[ks][e]), static_cast<float>(fg[ks][e]), dl);
    dl += __shfl_xor(dl, 32);
  }
  const float lse = q < a.seq ? a.lse[st_row] : INFINITY;
  if (lane < 32 && q < a.seq) a.delta[st_row] = dl;
  f32x16_t acc[HD / 32];
#pragma unroll
  for (int i = 0; i < HD / 32; ++i) zero(acc[i]);
  const int nt = (min(col0 + kAtCols, a.seq) + kAtTile - 1) / kAtTile;
  Tile<HD, true, TF32> tk;
  Tile<HD, false, TF32> tv;
  tk.load(a, base + d, a.ld, 0, tid);
  tv.load(a, base + 2 * d, a.ld, 0, tid);
  for (int t = 0; t < nt; ++t) {
    tk.store(lk, tid);
    tv.store(lv, tid);
    __syncthreads();
    if (t + 1 < nt) {
      tk.load(a, base + d, a.ld, (t + 1) * kAtTile, tid);
      tv.load(a, base + 2 * d, a.ld, (t + 1) * kAtTile, tid);
    }
    const int k0 = t * kAtTile;
    if (k0 <= q0 + 31 && q0 < a.seq) {
      const bool diag = k0 + kAtTile - 1 > q0;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        f32x16_t s, dp;
        zero(s);
        zero(dp);
#pragma unroll
        for (int ks = 0; ks < HD / 16; ++ks) {
          s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_rows<HD>(lk, 32 * kb, ks, lane), fq[ks], s, 0, 0, 0);
          dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_rows<HD>(lv, 32 * kb, ks, lane), fg[ks], dp, 0, 0, 0);
        }
        float ds[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = k0 + 32 * kb + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          const float p = diag && key > q ? 0.f : exp2f(s[r] * a.c2 - lse);
          ds[r] = p * (dp[r] - dl);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const bf16x8_t fd = pack8(ds + 8 * h);
#pragma unroll
          for (int i = 0; i < HD / 32; ++i)
            acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_cols<HD>(lk, 32 * i, 32 * kb + 16 * h, lane), fd,
                                                             acc[i], 0, 0, 0);
        }
      }
    }
    __syncthreads();
  }
  if (q < a.seq) store_own<HD, true, TF32>(a, acc, a.scale, a.dqkv + (tok0 + q) * a.ld + head * HD, q, lane);
}

// dK and dV: the wave's keys against every query tile that sees them (two
// products more than dQ, and the recomputed scores).
template <int HD, bool TF32>
__global__ __launch_bounds__(kAtThreads) void attn_bwd_kv_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(1024))) char lq[kAtTile * HD * 2];
  __shared__ __attribute__((aligned(1024))) char lg[kAtTile * HD * 2];
  __shared__ __attribute__((aligned(16))) float lst[2][kAtTile];  // lse, delta of the tile's queries
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int head = blockIdx.y, b = blockIdx.z, d = a.heads * HD;
  const int col0 = static_cast<int>(blockIdx.x) * kAtCols;
  const int key0 = col0 + 32 * wave, key = key0 + (lane & 31);
  const int64_t tok0 = static_cast<int64_t>(b) * a.seq;
  const uint16_t* base = a.qkv + tok0 * a.ld + head * HD;
  const uint16_t* go = a.go + tok0 * d + head * HD;
  const int64_t st0 = (static_cast<int64_t>(b) * a.heads + head) * a.seq;
  bf16x8_t fk[HD / 16], fv[HD / 16];
  load_own<HD, true, TF32>(a, base + d, a.ld, key, lane, fk);
  load_own<HD, false, TF32>(a, base + 2 * d, a.ld, key, lane, fv);
  f32x16_t dk[HD / 32], dv[HD / 32];
#pragma unroll
  for (int i = 0; i < HD / 32; ++i) {
    zero(dk[i]);
    zero(dv[i]);
  }
  const int t0 = col0 / kAtTile, nt = (a.seq + kAtTile - 1) / kAtTile;
  Tile<HD, true, TF32> tq;
  Tile<HD, false, TF32> tg;
  float st = 0.f;  // thread t < 128: lse (t < 64) or delta of the tile's query t % 64
  auto load_st = [&](int t) {
    const int r = t * kAtTile + (tid & 63);
    if (tid < 64) st = r < a.seq ? a.lse[st0 + r] : INFINITY;
    else if (tid < 128) st = r < a.seq ? a.delta[st0 + r] : 0.f;
  };
  tq.load(a, base, a.ld, t0 * kAtTile, tid);
  tg.load(a, go, d, t0 * kAtTile, tid);
  load_st(t0);
  for (int t = t0; t < nt; ++t) {
    tq.store(lq, tid);
    tg.store(lg, tid);
    if (tid < 128) lst[tid >> 6][tid & 63] = st;
    __syncthreads();
    if (t + 1 < nt) {
      tq.load(a, base, a.ld, (t + 1) * kAtTile, tid);
      tg.load(a, go, d, (t + 1) * kAtTile, tid);
      load_st(t + 1);
    }
    const int r0 = t * kAtTile;
    if (r0 + kAtTile - 1 >= key0 && key0 < a.seq) {  // wave-uniform: some query of the tile sees a key
      const bool diag = r0 < key0 + 31;
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        f32x16_t s, dp;
        zero(s);
        zero(dp);
#pragma unroll
        for (int ks = 0; ks < HD / 16; ++ks) {
          s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_rows<HD>(lq, 32 * qb, ks, lane), fk[ks], s, 0, 0, 0);
          dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_rows<HD>(lg, 32 * qb, ks, lane), fv[ks], dp, 0, 0, 0);
        }
        float p[16], ds[16];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int r = 32 * qb + 8 * g + 4 * (lane >> 5);
          const float4 ls = *reinterpret_cast<const float4*>(&lst[0][r]);
          const float4 de = *reinterpret_cast<const float4*>(&lst[1][r]);
          const float lsv[4] = {ls.x, ls.y, ls.z, ls.w}, dev[4] = {de.x, de.y, de.z, de.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x = diag && r0 + r + e < key ? 0.f : exp2f(s[4 * g + e] * a.c2 - lsv[e]);
            p[4 * g + e] = x;
            ds[4 * g + e] = x * (dp[4 * g + e] - dev[e]);
          }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const bf16x8_t fp = pack8(p + 8 * h), fd = pack8(ds + 8 * h);
#pragma unroll
          for (int i = 0; i < HD / 32; ++i) {
            dv[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_cols<HD>(lg, 32 * i, 32 * qb + 16 * h, lane), fp,
                                                            dv[i], 0, 0, 0);
            dk[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_cols<HD>(lq, 32 * i, 32 * qb + 16 * h, lane), fd,
                                                            dk[i], 0, 0, 0);
          }
        }
      }
    }
    __syncthreads();
  }
  if (key >= a.seq) return;
  uint16_t* dst = a.dqkv + (tok0 + key) * a.ld + head * HD;
  store_own<HD, true, TF32>(a, dk, a.scale, dst + d, key, lane);
  store_own<HD, false, TF32>(a, dv, 1.0f, dst + 2 * d, 0, lane);
}

// 128 keys a tile for sequences of 129 to 256 in heads of 64 (two tiles where
// 64 would take four; 4096 tokens of 256, 16 heads: 20.3 us, tiles of 64 20.6;
// the reason is the rounding, above), else 64.
template <int HD, bool TF32>
void launch_fwd(const AttnArgs& a, dim3 grid, hipStream_t st) {
  if constexpr (HD == 64) {
    if (a.seq > 128 && a.seq <= 256) {
      attn_fwd_kernel<HD, TF32, 128><<<grid, kAtThreads, 0, st>>>(a);
      return;
    }
  }
  attn_fwd_kernel<HD, TF32, 64><<<grid, kAtThreads, 0, st>>>(a);
}
template <int HD, bool TF32>
void launch_bwd_q(const AttnArgs& a, dim3 grid, hipStream_t st) {
  attn_bwd_q_kernel<HD, TF32><<<grid, kAtThreads, 0, st>>>(a);
}
template <int HD, bool TF32>
void launch_bwd_kv(const AttnArgs& a, dim3 grid, hipStream_t st) {
  attn_bwd_kv_kernel<HD, TF32><<<grid, kAtThreads, 0, st>>>(a);
}

int attn_check(const char* name, int64_t batch, int64_t seq, int64_t heads, int64_t head_dim, const void* qkv,
               int64_t ld, const void* cos, const void* sin, int table_dtype) {
  MOC_REQUIRE(batch >= 1 && seq >= 1 && heads >= 1 && batch <= 65535 && heads <= 65535 && seq < (1 << 24),
              "%s: bad shape", name);
  MOC_REQUIRE(head_dim == 64 || head_dim == 128, "%s: head_dim must be 64 or 128", name);
  MOC_REQUIRE(table_dtype == MOC_BF16 || table_dtype == MOC_F32, "%s: cos/sin must be bf16 or f32", name);
  MOC_REQUIRE(qkv != nullptr && aligned16(qkv) && ld % 8 == 0 && ld >= 3 * heads * head_dim,
              "%s: qkv needs 16-byte aligned rows of 3 heads head_dim", name);
  MOC_REQUIRE(cos != nullptr && sin != nullptr && aligned16(cos) && aligned16(sin), "%s: unaligned cos/sin", name);
  return MOC_OK;
}

}  // namespace
}  // namespace moc

using namespace moc;

#define MOC_ATTN_LAUNCH(LAUNCH)               \
  do {                                        \
    const bool tf = table_dtype == MOC_F32;   \
    if (head_dim == 64) {                     \
      if (tf) LAUNCH<64, true>(a, grid, st);  \
      else LAUNCH<64, false>(a, grid, st);    \
    } else {                                  \
      if (tf) LAUNCH<128, true>(a, grid, st); \
      else LAUNCH<128, false>(a, grid, st);   \
    }                                         \
  } while (0)

extern "C" int moc_rope_attention_forward_bf16(int64_t batch, int64_t seq, int64_t heads, int64_t head_dim,
                                               const void* qkv, int64_t ld, const void* cos, const void* sin,
                                               int table_dtype, float scale, void* o, float* lse, void* stream) {
  int rc = attn_check("moc_rope_attention_forward_bf16", batch, seq, heads, head_dim, qkv, ld, cos, sin, table_dtype);
  if (rc != MOC_OK) return rc;
  MOC_REQUIRE(o != nullptr && lse != nullptr && aligned16(o), "moc_rope_attention_forward_bf16: null or unaligned output");
  AttnArgs a{};
  a.qkv = static_cast<const uint16_t*>(qkv);
  a.ld = ld;
  a.heads = static_cast<int>(heads);
  a.seq = static_cast<int>(seq);
  a.cos = cos;
  a.sin = sin;
  a.scale = scale;
  a.c2 = scale * 1.44269504088896341f;
  a.o = static_cast<uint16_t*>(o);
  a.lse = lse;
  const dim3 grid(static_cast<unsigned>((seq + kAtCols - 1) / kAtCols), static_cast<unsigned>(heads),
                  static_cast<unsigned>(batch));
  hipStream_t st = as_stream(stream);
  MOC_ATTN_LAUNCH(launch_fwd);
  return check_launch("attn_fwd_kernel");
}

extern "C" int moc_rope_attention_backward_bf16(int64_t batch, int64_t seq, int64_t heads, int64_t head_dim,
                                                const void* qkv, int64_t ld, const void* cos, const void* sin,
                                                int table_dtype, float scale, const void* o, const float* lse,
                                                const void* go, float* delta, void* dqkv, void* stream) {
  int rc = attn_check("moc_rope_attention_backward_bf16", batch, seq, heads, head_dim, qkv, ld, cos, sin, table_dtype);
  if (rc != MOC_OK) return rc;
  MOC_REQUIRE(o && lse && go && delta && dqkv && aligned16(o) && aligned16(go) && aligned16(dqkv),
              "moc_rope_attention_backward_bf16: null or unaligned operand");
  AttnArgs a{};
  a.qkv = static_cast<const uint16_t*>(qkv);
  a.ld = ld;
  a.heads = static_cast<int>(heads);
  a.seq = static_cast<int>(seq);
  a.cos = cos;
  a.sin = sin;
  a.scale = scale;
  a.c2 = scale * 1.44269504088896341f;
  a.o = const_cast<uint16_t*>(static_cast<const uint16_t*>(o));
  a.lse = const_cast<float*>(lse);
  a.go = static_cast<const uint16_t*>(go);
  a.delta = delta;
  a.dqkv = static_cast<uint16_t*>(dqkv);
  const dim3 grid(static_cast<unsigned>((seq + kAtCols - 1) / kAtCols), static_cast<unsigned>(heads),
                  static_cast<unsigned>(batch));
  hipStream_t st = as_stream(stream);
  MOC_ATTN_LAUNCH(launch_bwd_q);
  rc = check_launch("attn_bwd_q_kernel");
  if (rc != MOC_OK) return rc;
  MOC_ATTN_LAUNCH(launch_bwd_kv);
  return check_launch("attn_bwd_kv_kernel");
}
