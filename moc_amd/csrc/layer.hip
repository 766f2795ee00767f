// The MoC FFN layer's forward (bf16 or f32) and backward (bf16) as one C-ABI
// call each: the launches of the single-stream path (moc/ffn.py:124-259 for `moc`,
// :262-369 for the 2:8 and post-SiLU selections, :372-497 for `moc_gcp`)
// issued from here instead of one host call per kernel.  At the shapes
// whose GEMMs fill the CUs about once (the 130m and 350m layers) the layer
// is host-bound otherwise: every Python wrapper and ctypes call costs
// microseconds that the GPU spends idle.
//
// No kernels of its own: the steps are the library's entry points, in the
// order of the reference's autograd Functions, on the caller's stream.
#include <algorithm>

#include "abi.h"

namespace {

int64_t gemm_ws(int64_t M, int64_t N, int64_t K, int64_t K2, int dt = MOC_BF16) {
  const int64_t b = moc_gemm_workspace_size(dt, M, N, K, K2);
  return b > 0 ? b : 0;
}

int64_t effective_2of8(int64_t inter) { return (inter / 8) * 2 + std::min<int64_t>(2, inter % 8); }

// 16-byte aligned rows of at least `cols` elements of `esz` bytes
bool ld_ok(const void* p, int64_t ld, int64_t cols, int64_t esz = 2) {
  return p != nullptr && moc::aligned16(p) && (ld * esz) % 16 == 0 && ld >= cols;
}

// The forward of moc_ffn_forward_bf16 / moc_ffn_forward_f32 in element type
// dt: G and U (one launch), the selection, the sparse aux, D.
int ffn_forward(int dt, const char* name, int64_t rows, int64_t d, int64_t inter, int64_t k, int selection,
                const void* x, int64_t ldx, const void* wg, int64_t ldwg, const void* wu, int64_t ldwu,
                const void* wd, int64_t ldwd, void* g, void* u, int64_t ld_gu, void* vals, void* idx,
                int idx_dtype, void* u_s, void* s_s, void* z_s, void* out, int64_t ldo, void* workspace,
                int64_t workspace_bytes, void* stream, const void* res = nullptr, int64_t ldres = 0) {
  const int64_t esz = dt == MOC_BF16 ? 2 : 4;
  MOC_REQUIRE(rows >= 1 && d >= 1 && inter >= 1 && k >= 1 && k <= inter, "%s: bad shape", name);
  MOC_REQUIRE(selection >= 0 && selection <= 2, "%s: selection 0 (Top-K), 1 (Top-K of |SiLU(G)|) or 2 (top-2 of 8)",
              name);
  MOC_REQUIRE(selection != 2 || k == effective_2of8(inter), "%s: the 2:8 selection keeps %lld channels", name,
              (long long)effective_2of8(inter));
  MOC_REQUIRE(ld_ok(x, ldx, d, esz) && ld_ok(wg, ldwg, d, esz) && ld_ok(wu, ldwu, d, esz) &&
                  ld_ok(wd, ldwd, inter, esz) && ld_ok(g, ld_gu, inter, esz) && ld_ok(u, ld_gu, inter, esz) &&
                  ld_ok(out, ldo, d, esz),
              "%s: operands need 16-byte aligned rows (leading dimensions multiples of %lld)", name,
              (long long)(16 / esz));
  MOC_REQUIRE(vals && idx && u_s, "%s: null output", name);
  const int64_t need = dt == MOC_BF16 ? moc_ffn_forward_workspace_size(rows, d, inter)
                                      : moc_ffn_forward_f32_workspace_size(rows, d, inter);
  MOC_REQUIRE(workspace_bytes >= need && (need == 0 || workspace != nullptr),
              "%s: workspace of %lld bytes required", name, (long long)need);
  // G = x Wg^T and U = x Wu^T (one launch)
  int rc;
  if (dt == MOC_BF16) {
    rc = moc_gemm_pair(rows, d, x, ldx, wg, ldwg, inter, g, ld_gu, wu, ldwu, inter, u, ld_gu, workspace,
                       workspace_bytes, stream);
  } else {
    rc = ldwg == ldwu ? moc::f32_gemm_pair(rows, inter, d, static_cast<const float*>(x), ldx,
                                           static_cast<const float*>(wg), static_cast<const float*>(wu), ldwg,
                                           static_cast<float*>(g), static_cast<float*>(u), ld_gu,
                                           moc::as_stream(stream))
                      : 1;
    if (rc == 1) {  // two launches
      rc = moc_gemm_ws(dt, rows, inter, d, x, ldx, 1, wg, 1, ldwg, 0, nullptr, 0, 0, nullptr, 0, 0, g, ld_gu, dt,
                       workspace, workspace_bytes, stream);
      if (rc == MOC_OK)
        rc = moc_gemm_ws(dt, rows, inter, d, x, ldx, 1, wu, 1, ldwu, 0, nullptr, 0, 0, nullptr, 0, 0, u, ld_gu,
                         dt, workspace, workspace_bytes, stream);
    }
  }
  if (rc != MOC_OK) return rc;
  // the selection (indices in ascending channel order) and its gate values
  if (selection == 2)
    rc = moc_select_2of8(dt, g, rows, inter, ld_gu, vals, idx, idx_dtype, stream);
  else
    rc = moc_topk_rows(dt, g, rows, inter, ld_gu, k, selection, vals, idx, idx_dtype, nullptr, 0, stream);
  if (rc != MOC_OK) return rc;
  // U at the selection, SiLU, Z; the dense zero-filled Z goes into G's
  // buffer, which nothing reads after the selection
  rc = moc_sparse_forward_aux(dt, vals, idx, idx_dtype, u, ld_gu, rows, k, inter, u_s, s_s, z_s, g, ld_gu,
                              stream);
  if (rc != MOC_OK) return rc;
  // D = Z W_down^T (with a residual: res + D from the same epilogue)
  if (res != nullptr)
    return moc_gemm_residual_bf16(rows, d, inter, g, ld_gu, 1, wd, 1, ldwd, out, ldo, res, ldres, workspace,
                                  workspace_bytes, stream);
  return moc_gemm_ws(dt, rows, d, inter, g, ld_gu, 1, wd, 1, ldwd, 0, nullptr, 0, 0, nullptr, 0, 0, out, ldo, dt,
                     workspace, workspace_bytes, stream);
}

}  // namespace

// ---------------------------------------------------------------------------
// Inference of one MoC FFN layer for more tokens than the decode kernels take
// (moc/inference/inference_ffn.py:169-203): G and U on the MFMA GEMM (one
// launch), the selection, the dense Z, y = Z W_down from the module's
// W_down^T.  From 17 tokens on a token's selected rows of W_up and W_down
// overlap the other tokens' so much that reading both weights once, densely,
// beats gathering rows token by token: 200 tokens of 2048 -> 5461, K 1024:
// 214 us in the gathered Up and Down alone (245 the layer), 48 here for the layer.
// Scratch: G and U (rows of `pitch`), the selected gate values and indices;
// Z takes G's place.
// ---------------------------------------------------------------------------
namespace {
struct InferScratch {
  int64_t pitch, g, u, vals, idx, bytes;
};
InferScratch infer_scratch(int64_t rows, int64_t inter, int64_t k, int selection) {
  auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
  InferScratch s;
  s.pitch = inter >= 512 ? (inter + 63) / 64 * 64 : (inter + 7) / 8 * 8;
  s.g = 0;
  s.u = up(rows * s.pitch * 2);
  s.vals = 2 * s.u;
  s.idx = s.vals + (selection == 0 ? up(rows * k * 2) : 0);
  s.bytes = s.idx + (selection == 0 ? up(rows * k * 2) : 0);
  return s;
}
}  // namespace

extern "C" int64_t moc_ffn_infer_scratch_size(int64_t rows, int64_t inter, int64_t k, int selection) {
  if (rows <= 0 || inter <= 0 || k <= 0) return 0;
  return infer_scratch(rows, inter, k, selection).bytes;
}

extern "C" int64_t moc_ffn_infer_workspace_size(int64_t rows, int64_t d, int64_t inter) {
  if (rows <= 0 || d <= 0 || inter <= 0) return 0;
  return std::max(gemm_ws(rows, inter, d, 0), gemm_ws(rows, d, inter, 0));
}

extern "C" int moc_ffn_infer_bf16(int64_t rows, int64_t d, int64_t inter, int64_t k, int selection, const void* x,
                                  int64_t ldx, const void* wg, const void* wu, const void* wdt, int64_t ldwdt,
                                  const void* res, int64_t ldres, void* y, int64_t ldy, void* scratch,
                                  int64_t scratch_bytes, void* workspace, int64_t workspace_bytes, void* stream) {
  MOC_REQUIRE(rows >= 1 && d >= 8 && d % 8 == 0 && inter >= 1 && k >= 1 && k <= inter, "moc_ffn_infer_bf16: bad shape");
  MOC_REQUIRE(selection == 0 || (selection == 2 && inter % 8 == 0 && k == effective_2of8(inter)),
              "moc_ffn_infer_bf16: selection 0 (Top-K) or 2 (top-2 of 8, intermediate a multiple of 8)");
  MOC_REQUIRE(inter <= 32768, "moc_ffn_infer_bf16: intermediate size above 32768");
  MOC_REQUIRE(ld_ok(x, ldx, d) && ld_ok(wg, d, d) && ld_ok(wu, d, d) && ld_ok(wdt, ldwdt, d) && ld_ok(y, ldy, d) &&
                  (res == nullptr || ld_ok(res, ldres, d)),
              "moc_ffn_infer_bf16: operands need 16-byte aligned rows");
  const InferScratch s = infer_scratch(rows, inter, k, selection);
  MOC_REQUIRE(scratch != nullptr && moc::aligned16(scratch) && scratch_bytes >= s.bytes,
              "moc_ffn_infer_bf16: scratch of %lld bytes required", (long long)s.bytes);
  const int64_t need = moc_ffn_infer_workspace_size(rows, d, inter);
  MOC_REQUIRE(workspace_bytes >= need && (need == 0 || workspace != nullptr),
              "moc_ffn_infer_bf16: workspace of %lld bytes required", (long long)need);
  char* base = static_cast<char*>(scratch);
  void *g = base + s.g, *u = base + s.u, *vals = base + s.vals, *idx = base + s.idx;
  int rc = moc_gemm_pair(rows, d, x, ldx, wg, d, inter, g, s.pitch, wu, d, inter, u, s.pitch, workspace,
                         workspace_bytes, stream);
  if (rc != MOC_OK) return rc;
  if (selection == 2) {
    rc = moc::select28_dense(g, u, s.pitch, rows, inter, moc::as_stream(stream));
  } else {
    rc = moc_topk_rows(MOC_BF16, g, rows, inter, s.pitch, k, 0, vals, idx, MOC_I16, nullptr, 0, stream);
    if (rc == MOC_OK)
      rc = moc_sparse_forward_aux(MOC_BF16, vals, idx, MOC_I16, u, s.pitch, rows, k, inter, nullptr, nullptr,
                                  nullptr, g, s.pitch, stream);
  }
  if (rc != MOC_OK) return rc;
  if (res != nullptr)
    return moc_gemm_residual_bf16(rows, d, inter, g, s.pitch, 1, wdt, ldwdt, 1, y, ldy, res, ldres, workspace,
                                  workspace_bytes, stream);
  return moc_gemm_ws(MOC_BF16, rows, d, inter, g, s.pitch, 1, wdt, ldwdt, 1, 0, nullptr, 0, 0, nullptr, 0, 0, y, ldy,
                     MOC_BF16, workspace, workspace_bytes, stream);
}

// GEMM workspace of moc_ffn_forward_bf16: the G,U pair and D = Z W_down^T.
extern "C" int64_t moc_ffn_forward_workspace_size(int64_t rows, int64_t d, int64_t inter) {
  if (rows <= 0 || d <= 0 || inter <= 0) return 0;
  return std::max(gemm_ws(rows, inter, d, 0), gemm_ws(rows, d, inter, 0));
}

// GEMM workspace of moc_ffn_forward_f32: G and U when they run as two
// launches, and D = Z W_down^T.
extern "C" int64_t moc_ffn_forward_f32_workspace_size(int64_t rows, int64_t d, int64_t inter) {
  if (rows <= 0 || d <= 0 || inter <= 0) return 0;
  return std::max(gemm_ws(rows, inter, d, 0, MOC_F32), gemm_ws(rows, d, inter, 0, MOC_F32));
}

extern "C" int moc_ffn_forward_bf16(int64_t rows, int64_t d, int64_t inter, int64_t k, int selection,
                                    const void* x, int64_t ldx, const void* wg, int64_t ldwg,
                                    const void* wu, int64_t ldwu, const void* wd, int64_t ldwd, void* g,
                                    void* u, int64_t ld_gu, void* vals, void* idx, int idx_dtype,
                                    void* u_s, void* s_s, void* z_s, void* out, int64_t ldo,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
  return ffn_forward(MOC_BF16, "moc_ffn_forward_bf16", rows, d, inter, k, selection, x, ldx, wg, ldwg, wu, ldwu,
                     wd, ldwd, g, u, ld_gu, vals, idx, idx_dtype, u_s, s_s, z_s, out, ldo, workspace,
                     workspace_bytes, stream);
}

extern "C" int moc_ffn_forward_f32(int64_t rows, int64_t d, int64_t inter, int64_t k, int selection,
                                   const void* x, int64_t ldx, const void* wg, int64_t ldwg, const void* wu,
                                   int64_t ldwu, const void* wd, int64_t ldwd, void* g, void* u, int64_t ld_gu,
                                   void* vals, void* idx, int idx_dtype, void* u_s, void* s_s, void* z_s,
                                   void* out, int64_t ldo, void* workspace, int64_t workspace_bytes,
                                   void* stream) {
  return ffn_forward(MOC_F32, "moc_ffn_forward_f32", rows, d, inter, k, selection, x, ldx, wg, ldwg, wu, ldwu,
                     wd, ldwd, g, u, ld_gu, vals, idx, idx_dtype, u_s, s_s, z_s, out, ldo, workspace,
                     workspace_bytes, stream);
}

// GEMM workspace of moc_ffn_backward_bf16 (stacked: dWg and dWu as one GEMM
// over [gG | gU] with rows ld_ggu / 2 apart).
extern "C" int64_t moc_ffn_backward_workspace_size(int64_t rows, int64_t d, int64_t inter, int64_t ld_ggu,
                                                   int stacked) {
  if (rows <= 0 || d <= 0 || inter <= 0) return 0;
  int64_t w = std::max(gemm_ws(d, inter, rows, 0), gemm_ws(rows, inter, d, 0));
  w = std::max(w, stacked ? gemm_ws(ld_ggu, d, rows, 0) : gemm_ws(inter, d, rows, 0));
  if (stacked) w = std::max(w, moc::gemm_split_pair_workspace(ld_ggu, d, rows, d, inter, rows));
  return std::max(w, gemm_ws(rows, d, inter, inter));
}

extern "C" int moc_ffn_backward_bf16(int64_t rows, int64_t d, int64_t inter, int64_t k, const void* go,
                                     int64_t ldgo, const void* x, int64_t ldx, const void* idx, int idx_dtype,
                                     const void* g_s, const void* u_s, const void* s_s, const void* z_s,
                                     const void* wg, int64_t ldwg, const void* wu, int64_t ldwu,
                                     const void* wd, int64_t ldwd, void* zbuf, int64_t ldz, void* gg, void* gu,
                                     int64_t ld_ggu, int stacked, void* s_tmp, void* dx, int64_t lddx,
                                     void* dwg, void* dwu, int64_t ld_dw, void* dwd, int64_t lddwd,
                                     int grad_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  MOC_REQUIRE(rows >= 1 && d >= 1 && inter >= 1 && k >= 1 && k <= inter, "moc_ffn_backward_bf16: bad shape");
  MOC_REQUIRE(grad_dtype == MOC_BF16 || grad_dtype == MOC_F32, "moc_ffn_backward_bf16: grad dtype bf16 or f32");
  MOC_REQUIRE(ld_ok(go, ldgo, d) && ld_ok(x, ldx, d) && ld_ok(wg, ldwg, d) && ld_ok(wu, ldwu, d) &&
                  ld_ok(wd, ldwd, inter) && ld_ok(zbuf, ldz, inter) && ld_ok(gg, ld_ggu, inter) &&
                  ld_ok(gu, ld_ggu, inter) && ld_ok(dx, lddx, d),
              "moc_ffn_backward_bf16: operands need 16-byte aligned rows (leading dimensions multiples of 8)");
  MOC_REQUIRE(idx && g_s && u_s && dwg && dwu && dwd && ld_dw >= d && lddwd >= inter,
              "moc_ffn_backward_bf16: null operand or bad leading dimension");
  MOC_REQUIRE(s_s == nullptr || z_s != nullptr, "moc_ffn_backward_bf16: saved S needs saved Z");
  const int64_t esz = grad_dtype == MOC_BF16 ? 2 : 4;
  const int64_t pitch = ld_ggu / 2;
  if (stacked) {
    MOC_REQUIRE(ld_ggu % 16 == 0 && pitch >= inter &&
                    static_cast<const char*>(gu) == static_cast<const char*>(gg) + pitch * 2 &&
                    static_cast<const char*>(dwu) == static_cast<const char*>(dwg) + pitch * ld_dw * esz,
                "moc_ffn_backward_bf16: stacked gG | gU and dWg | dWu must be one buffer each, pitch apart");
  }
  const int64_t need = moc_ffn_backward_workspace_size(rows, d, inter, ld_ggu, stacked);
  MOC_REQUIRE(workspace_bytes >= need && (need == 0 || workspace != nullptr),
              "moc_ffn_backward_bf16: workspace of %lld bytes required", (long long)need);
  // Stacked layout within the row kernels' limits: gZ goes into gU's rows,
  // the gradient pass turns them into gG | gU in place and writes the dense
  // Z as well (no scatter launch), so Z outlives gZ and the weight gradients
  // run last, dWd beside [dWg | dWu] as one grouped split-K launch where
  // both split K.
  const bool late = stacked && ld_ggu <= 8192 && ldz <= 8192 && moc::aligned16(gu);
  hipStream_t st = moc::as_stream(stream);
  int rc;
  if (late) {
    // gZ = go W_down into gU's rows
    rc = moc_gemm_ws(MOC_BF16, rows, inter, d, go, ldgo, 1, wd, ldwd, 1, 0, nullptr, 0, 0, nullptr, 0, 0, gu,
                     ld_ggu, MOC_BF16, workspace, workspace_bytes, stream);
    if (rc != MOC_OK) return rc;
    // gG, gU dense (:455-480) and Z (GCP: S, Z recomputed, :435-437)
    rc = 1;
    if (s_s != nullptr || s_tmp == nullptr) {
      rc = moc::sparse_backward_aux_z(idx, idx_dtype, g_s, u_s, s_s, s_s != nullptr ? z_s : nullptr, gu, ld_ggu,
                                      rows, k, inter, gg, gu, ld_ggu, zbuf, ldz, st);
      if (rc < 0) return rc;
    }
    if (rc == 1) {  // S wanted in s_tmp, or no fused form: the scatter, then gG | gU in place
      rc = s_s == nullptr
               ? moc_gcp_recompute_scatter(MOC_BF16, g_s, u_s, idx, idx_dtype, rows, k, inter, s_tmp, zbuf, ldz,
                                           stream)
               : moc_scatter_sparse_to_dense(MOC_BF16, z_s, idx, idx_dtype, rows, k, inter, zbuf, ldz, stream);
      if (rc != MOC_OK) return rc;
      rc = moc_sparse_backward_aux(MOC_BF16, idx, idx_dtype, g_s, u_s, s_s, gu, ld_ggu, rows, k, inter, gg, gu,
                                   ld_ggu, stream);
    }
    if (rc != MOC_OK) return rc;
    // [dWg | dWu] = [gG | gU]^T x (:483-490) and dWd = go^T Z (:447): one
    // grouped launch where the plan takes them, else two
    const int64_t pair_ws = moc::gemm_split_pair_workspace(2 * pitch, d, rows, d, inter, rows);
    rc = 1;
    if (pair_ws > 0 && workspace_bytes >= pair_ws)
      rc = moc::gemm_split_pair(2 * pitch, d, rows, gg, 1, ld_ggu, x, ldx, 1, dwg, ld_dw, d, inter, rows, go, 1,
                                ldgo, zbuf, ldz, 1, dwd, lddwd, grad_dtype, workspace, workspace_bytes, st);
    if (rc == 1) {
      rc = moc_gemm_ws(MOC_BF16, 2 * pitch, d, rows, gg, 1, ld_ggu, x, ldx, 1, 0, nullptr, 0, 0, nullptr, 0, 0,
                       dwg, ld_dw, grad_dtype, workspace, workspace_bytes, stream);
      if (rc == MOC_OK)
        rc = moc_gemm_ws(MOC_BF16, d, inter, rows, go, 1, ldgo, zbuf, ldz, 1, 0, nullptr, 0, 0, nullptr, 0, 0,
                         dwd, lddwd, grad_dtype, workspace, workspace_bytes, stream);
    }
    if (rc != MOC_OK) return rc;
    // dX = gG Wg + gU Wu (:491-497)
    return moc_gemm_ws(MOC_BF16, rows, d, inter, gg, ld_ggu, 1, wg, ldwg, 1, inter, gu, ld_ggu, 1, wu, ldwu, 1,
                       dx, lddx, MOC_BF16, workspace, workspace_bytes, stream);
  }
  if (s_s == nullptr) {
    // GCP: S = SiLU(G M), Z = S U M recomputed, Z scattered dense (:435-442)
    rc = moc_gcp_recompute_scatter(MOC_BF16, g_s, u_s, idx, idx_dtype, rows, k, inter, s_tmp, zbuf, ldz, stream);
  } else {
    rc = moc_scatter_sparse_to_dense(MOC_BF16, z_s, idx, idx_dtype, rows, k, inter, zbuf, ldz, stream);
  }
  if (rc != MOC_OK) return rc;
  // dWd = go^T Z
  rc = moc_gemm_ws(MOC_BF16, d, inter, rows, go, 1, ldgo, zbuf, ldz, 1, 0, nullptr, 0, 0, nullptr, 0, 0, dwd,
                   lddwd, grad_dtype, workspace, workspace_bytes, stream);
  if (rc != MOC_OK) return rc;
  // gZ = go W_down, into Z's buffer (Z is consumed)
  rc = moc_gemm_ws(MOC_BF16, rows, inter, d, go, ldgo, 1, wd, ldwd, 1, 0, nullptr, 0, 0, nullptr, 0, 0, zbuf,
                   ldz, MOC_BF16, workspace, workspace_bytes, stream);
  if (rc != MOC_OK) return rc;
  // gG, gU dense (:455-480); GCP: the kernel recomputes S from g_s (the
  // same bits as the recompute above)
  rc = moc_sparse_backward_aux(MOC_BF16, idx, idx_dtype, g_s, u_s, s_s, zbuf, ldz, rows, k, inter, gg, gu,
                               ld_ggu, stream);
  if (rc != MOC_OK) return rc;
  // dWg = gG^T x, dWu = gU^T x (:483-490)
  if (stacked) {
    rc = moc_gemm_ws(MOC_BF16, 2 * pitch, d, rows, gg, 1, ld_ggu, x, ldx, 1, 0, nullptr, 0, 0, nullptr, 0, 0,
                     dwg, ld_dw, grad_dtype, workspace, workspace_bytes, stream);
  } else {
    rc = moc_gemm_ws(MOC_BF16, inter, d, rows, gg, 1, ld_ggu, x, ldx, 1, 0, nullptr, 0, 0, nullptr, 0, 0, dwg,
                     ld_dw, grad_dtype, workspace, workspace_bytes, stream);
    if (rc != MOC_OK) return rc;
    rc = moc_gemm_ws(MOC_BF16, inter, d, rows, gu, 1, ld_ggu, x, ldx, 1, 0, nullptr, 0, 0, nullptr, 0, 0, dwu,
                     ld_dw, grad_dtype, workspace, workspace_bytes, stream);
  }
  if (rc != MOC_OK) return rc;
  // dX = gG Wg + gU Wu (:491-497)
  return moc_gemm_ws(MOC_BF16, rows, d, inter, gg, ld_ggu, 1, wg, ldwg, 1, inter, gu, ld_ggu, 1, wu, ldwu, 1, dx,
                     lddx, MOC_BF16, workspace, workspace_bytes, stream);
}

// ---------------------------------------------------------------------------
// The FFN half of a pre-norm decoder block, h + FFN(RMSNorm(h))
// (moc/model.py:20-28,83-86), as one call per pass: the norm as a row pass,
// the FFN's launches, the residual add in the Down GEMM's epilogue; the
// backward recomputes the norm's output (same kernel, same bits) instead of
// keeping it, runs the FFN backward and then the norm's backward with the
// residual branch's gradient added.

extern "C" int moc_ffn_block_forward_bf16(int64_t rows, int64_t d, int64_t inter, int64_t k, int selection,
                                          const void* h, int64_t ldh, const void* norm_w, float eps, void* xn,
                                          int64_t ldxn, float* rstd, const void* wg, int64_t ldwg, const void* wu,
                                          int64_t ldwu, const void* wd, int64_t ldwd, void* g, void* u,
                                          int64_t ld_gu, void* vals, void* idx, int idx_dtype, void* u_s,
                                          void* s_s, void* z_s, void* out, int64_t ldo, void* workspace,
                                          int64_t workspace_bytes, void* stream) {
  MOC_REQUIRE(rstd != nullptr, "moc_ffn_block_forward_bf16: null rstd");
  MOC_REQUIRE(ld_ok(h, ldh, d), "moc_ffn_block_forward_bf16: h needs 16-byte aligned rows");
  int rc = moc_rmsnorm_rows_bf16(h, ldh, rows, d, norm_w, eps, xn, ldxn, rstd, stream);
  if (rc != MOC_OK) return rc;
  return ffn_forward(MOC_BF16, "moc_ffn_block_forward_bf16", rows, d, inter, k, selection, xn, ldxn, wg, ldwg, wu,
                     ldwu, wd, ldwd, g, u, ld_gu, vals, idx, idx_dtype, u_s, s_s, z_s, out, ldo, workspace,
                     workspace_bytes, stream, h, ldh);
}

namespace {
// Where the norm backward's partial rows start in the block backward's
// workspace: after the FFN backward's GEMM workspace, and never inside the
// GEMM arrival counters at its start (which must stay zero between calls).
int64_t block_rms_offset(int64_t rows, int64_t d, int64_t inter, int64_t ld_ggu, int stacked) {
  const int64_t f = (moc_ffn_backward_workspace_size(rows, d, inter, ld_ggu, stacked) + 255) / 256 * 256;
  return std::max<int64_t>(f, MOC_GEMM_WS_COUNTER_BYTES);
}
}  // namespace

extern "C" int64_t moc_ffn_block_backward_workspace_size(int64_t rows, int64_t d, int64_t inter, int64_t ld_ggu,
                                                         int stacked) {
  if (rows <= 0 || d <= 0 || inter <= 0) return 0;
  return block_rms_offset(rows, d, inter, ld_ggu, stacked) + moc_rmsnorm_backward_workspace_size(rows, d);
}

extern "C" int moc_ffn_block_backward_bf16(int64_t rows, int64_t d, int64_t inter, int64_t k, const void* dout,
                                           int64_t ldgo, const void* h, int64_t ldh, const void* norm_w, float eps,
                                           const float* rstd, void* xn, int64_t ldxn, const void* idx,
                                           int idx_dtype, const void* g_s, const void* u_s, const void* s_s,
                                           const void* z_s, const void* wg, int64_t ldwg, const void* wu,
                                           int64_t ldwu, const void* wd, int64_t ldwd, void* zbuf, int64_t ldz,
                                           void* gg, void* gu, int64_t ld_ggu, int stacked, void* s_tmp,
                                           void* dh, int64_t lddh, void* dwg, void* dwu, int64_t ld_dw, void* dwd,
                                           int64_t lddwd, int grad_dtype, void* dnorm_w, int dnorm_dtype,
                                           void* workspace, int64_t workspace_bytes, void* stream) {
  MOC_REQUIRE(rows >= 1 && d >= 1, "moc_ffn_block_backward_bf16: bad shape");
  const int64_t need = moc_ffn_block_backward_workspace_size(rows, d, inter, ld_ggu, stacked);
  MOC_REQUIRE(workspace != nullptr && workspace_bytes >= need && moc::aligned16(workspace),
              "moc_ffn_block_backward_bf16: workspace of %lld bytes required", (long long)need);
  MOC_REQUIRE(ld_ok(h, ldh, d) && ld_ok(xn, ldxn, d) && ld_ok(dh, lddh, d) && rstd != nullptr,
              "moc_ffn_block_backward_bf16: h, xn and dh need 16-byte aligned rows");
  const int64_t f = block_rms_offset(rows, d, inter, ld_ggu, stacked);
  // the FFN's input again (the forward's row pass: same bits)
  int rc = moc_rmsnorm_rows_bf16(h, ldh, rows, d, norm_w, eps, xn, ldxn, nullptr, stream);
  if (rc != MOC_OK) return rc;
  // FFN backward; its dX (the norm output's gradient) goes into xn's buffer:
  // xn is last read by the weight-gradient GEMMs, which run before dX
  rc = moc_ffn_backward_bf16(rows, d, inter, k, dout, ldgo, xn, ldxn, idx, idx_dtype, g_s, u_s, s_s, z_s, wg,
                             ldwg, wu, ldwu, wd, ldwd, zbuf, ldz, gg, gu, ld_ggu, stacked, s_tmp, xn, ldxn, dwg,
                             dwu, ld_dw, dwd, lddwd, grad_dtype, workspace, f, stream);
  if (rc != MOC_OK) return rc;
  // dh = dout (the residual branch) + the norm's backward of dX
  return moc_rmsnorm_backward_bf16(h, ldh, rows, d, norm_w, rstd, xn, ldxn, dout, ldgo, dh, lddh, dnorm_w,
                                   dnorm_dtype, static_cast<char*>(workspace) + f, workspace_bytes - f, stream);
}

// ---------------------------------------------------------------------------
// The attention half of a block, x + out_proj(attention(RMSNorm(x)))
// (moc/model.py:31-64,83-84), as one call per pass, for a bf16 stream with
// bf16 weights or an f32 stream with f32 weights (bf16 autocast: the weights
// are cast here, one launch).  What the backward needs beyond x lives in one
// caller buffer, laid out here.

namespace {
struct AttnHalf {
  int64_t t, d, heads;
  // saved by the forward
  int64_t xn, qkv, o, rstd, lse, wq, wo, saved;
  // scratch of the backward: go (f32 stream), do / dxn, dqkv, delta, norm partials
  int64_t go, dox, dqkv, delta, rms, scratch;
};
AttnHalf attn_half(int64_t batch, int64_t seq, int64_t heads, int64_t head_dim, int f32) {
  auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
  AttnHalf a{};
  a.t = batch * seq;
  a.d = heads * head_dim;
  a.heads = heads;
  int64_t p = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = p;
    p += up(bytes);
    return at;
  };
  a.xn = take(a.t * a.d * 2);
  a.qkv = take(a.t * a.d * 6);
  a.o = take(a.t * a.d * 2);
  a.rstd = take(a.t * 4);
  a.lse = take(a.t * heads * 4);
  a.wq = take(f32 ? a.d * a.d * 6 : 0);
  a.wo = take(f32 ? a.d * a.d * 2 : 0);
  a.saved = p;
  p = 0;
  a.go = take(f32 ? a.t * a.d * 2 : 0);
  a.dox = take(a.t * a.d * 2);
  a.dqkv = take(a.t * a.d * 6);
  a.delta = take(a.t * heads * 4);
  a.rms = take(moc_rmsnorm_backward_workspace_size(a.t, a.d));
  a.scratch = p;
  return a;
}
bool attn_half_shape(int64_t batch, int64_t seq, int64_t heads, int64_t head_dim) {
  return batch >= 1 && seq >= 1 && batch * seq >= 2 && heads >= 1 && (head_dim == 64 || head_dim == 128) &&
         heads * head_dim <= 4096 && batch * seq < (1LL << 31);
}
}  // namespace

extern "C" int64_t moc_attention_half_saved_size(int64_t batch, int64_t seq, int64_t heads, int64_t head_dim, int f32) {
  return attn_half_shape(batch, seq, heads, head_dim) ? attn_half(batch, seq, heads, head_dim, f32).saved : 0;
}
extern "C" int64_t moc_attention_half_scratch_size(int64_t batch, int64_t seq, int64_t heads, int64_t head_dim,
                                                   int f32) {
  return attn_half_shape(batch, seq, heads, head_dim) ? attn_half(batch, seq, heads, head_dim, f32).scratch : 0;
}
extern "C" int64_t moc_attention_half_workspace_size(int64_t tokens, int64_t d) {
  if (tokens <= 0 || d <= 0) return 0;
  return std::max({gemm_ws(tokens, 3 * d, d, 0), gemm_ws(tokens, d, d, 0), gemm_ws(d, d, tokens, 0),
                   gemm_ws(3 * d, d, tokens, 0), gemm_ws(tokens, d, 3 * d, 0)});
}

extern "C" int moc_attention_half_forward(int64_t batch, int64_t seq, int64_t heads, int64_t head_dim, int f32,
                                          const void* x, const void* norm_w, float eps, const void* w_qkv,
                                          const void* w_out, const void* cos, const void* sin, float scale, void* h,
                                          void* saved, int64_t saved_bytes, void* y_tmp, void* workspace,
                                          int64_t workspace_bytes, void* stream) {
  MOC_REQUIRE(attn_half_shape(batch, seq, heads, head_dim),
              "moc_attention_half_forward: two tokens or more, heads of 64 or 128, hidden up to 4096");
  const AttnHalf a = attn_half(batch, seq, heads, head_dim, f32);
  const int64_t t = a.t, d = a.d;
  MOC_REQUIRE(x && norm_w && w_qkv && w_out && h && saved && (!f32 || y_tmp),
              "moc_attention_half_forward: null pointer");
  MOC_REQUIRE(moc::aligned16(x) && moc::aligned16(w_qkv) && moc::aligned16(w_out) && moc::aligned16(h) &&
                  moc::aligned16(saved) && moc::aligned16(y_tmp),
              "moc_attention_half_forward: operands must be 16-byte aligned");
  MOC_REQUIRE(saved_bytes >= a.saved, "moc_attention_half_forward: buffer of %lld bytes required", (long long)a.saved);
  const int64_t need = moc_attention_half_workspace_size(t, d);
  MOC_REQUIRE(workspace_bytes >= need && (need == 0 || workspace != nullptr),
              "moc_attention_half_forward: workspace of %lld bytes required", (long long)need);
  char* b = static_cast<char*>(saved);
  void *xn = b + a.xn, *qkv = b + a.qkv, *o = b + a.o;
  float *rstd = reinterpret_cast<float*>(b + a.rstd), *lse = reinterpret_cast<float*>(b + a.lse);
  const void *wq = w_qkv, *wo = w_out;
  int rc;
  if (f32) {
    const void* src[2] = {w_qkv, w_out};
    void* dst[2] = {b + a.wq, b + a.wo};
    const int64_t rows[2] = {3 * d, d}, cols[2] = {d, d};
    rc = moc_cast_bf16_multi(2, src, rows, cols, dst, cols, stream);
    if (rc != MOC_OK) return rc;
    wq = dst[0];
    wo = dst[1];
    rc = moc_rmsnorm_rows_f32(static_cast<const float*>(x), d, t, d, static_cast<const float*>(norm_w), eps, xn, d,
                              rstd, stream);
  } else {
    rc = moc_rmsnorm_rows_bf16(x, d, t, d, norm_w, eps, xn, d, rstd, stream);
  }
  if (rc != MOC_OK) return rc;
  rc = moc_gemm_ws(MOC_BF16, t, 3 * d, d, xn, d, 1, wq, 1, d, 0, nullptr, 0, 0, nullptr, 0, 0, qkv, 3 * d, MOC_BF16,
                   workspace, workspace_bytes, stream);
  if (rc != MOC_OK) return rc;
  rc = moc_rope_attention_forward_bf16(batch, seq, heads, head_dim, qkv, 3 * d, cos, sin, f32 ? MOC_F32 : MOC_BF16,
                                       scale, o, lse, stream);
  if (rc != MOC_OK) return rc;
  if (!f32)
    return moc_gemm_residual_bf16(t, d, d, o, d, 1, wo, 1, d, h, d, x, d, workspace, workspace_bytes, stream);
  rc = moc_gemm_ws(MOC_BF16, t, d, d, o, d, 1, wo, 1, d, 0, nullptr, 0, 0, nullptr, 0, 0, y_tmp, d, MOC_BF16,
                   workspace, workspace_bytes, stream);
  if (rc != MOC_OK) return rc;
  return moc::add_f32_bf16(static_cast<const float*>(x), y_tmp, static_cast<float*>(h), t * d,
                           moc::as_stream(stream));
}

extern "C" int moc_attention_half_backward(int64_t batch, int64_t seq, int64_t heads, int64_t head_dim, int f32,
                                           const void* dh, const void* x, const void* norm_w, const void* w_qkv,
                                           const void* w_out, const void* cos, const void* sin, float scale,
                                           const void* saved, int64_t saved_bytes, void* dx, void* dnorm_w,
                                           void* dw_qkv, void* dw_out, void* scratch, int64_t scratch_bytes,
                                           void* workspace, int64_t workspace_bytes, void* stream) {
  MOC_REQUIRE(attn_half_shape(batch, seq, heads, head_dim),
              "moc_attention_half_backward: two tokens or more, heads of 64 or 128, hidden up to 4096");
  const AttnHalf a = attn_half(batch, seq, heads, head_dim, f32);
  const int64_t t = a.t, d = a.d;
  MOC_REQUIRE(dh && x && norm_w && w_qkv && w_out && saved && scratch && (dx != nullptr) == (dnorm_w != nullptr),
              "moc_attention_half_backward: null pointer");
  if (dx == nullptr && dw_qkv == nullptr && dw_out == nullptr) return MOC_OK;
  MOC_REQUIRE(moc::aligned16(dh) && moc::aligned16(x) && moc::aligned16(w_qkv) && moc::aligned16(w_out) &&
                  moc::aligned16(saved) && moc::aligned16(dx) && moc::aligned16(scratch),
              "moc_attention_half_backward: operands must be 16-byte aligned");
  MOC_REQUIRE(saved_bytes >= a.saved && scratch_bytes >= a.scratch,
              "moc_attention_half_backward: buffers of %lld and %lld bytes required", (long long)a.saved,
              (long long)a.scratch);
  const int64_t need = moc_attention_half_workspace_size(t, d);
  MOC_REQUIRE(workspace_bytes >= need && (need == 0 || workspace != nullptr),
              "moc_attention_half_backward: workspace of %lld bytes required", (long long)need);
  const char* b = static_cast<const char*>(saved);
  char* s = static_cast<char*>(scratch);
  const void *xn = b + a.xn, *qkv = b + a.qkv, *o = b + a.o;
  const float *rstd = reinterpret_cast<const float*>(b + a.rstd), *lse = reinterpret_cast<const float*>(b + a.lse);
  const void *wq = f32 ? b + a.wq : w_qkv, *wo = f32 ? b + a.wo : w_out, *go = dh;
  void *dox = s + a.dox, *dqkv = s + a.dqkv;
  const int gdt = f32 ? MOC_F32 : MOC_BF16;
  int rc;
  if (f32) {
    const void* src[1] = {dh};
    void* dst[1] = {s + a.go};
    rc = moc_cast_bf16_multi(1, src, &t, &d, dst, &d, stream);
    if (rc != MOC_OK) return rc;
    go = dst[0];
  }
  // dW_out = go^T o
  if (dw_out != nullptr) {
    rc = moc_gemm_ws(MOC_BF16, d, d, t, go, 1, d, o, d, 1, 0, nullptr, 0, 0, nullptr, 0, 0, dw_out, d, gdt, workspace,
                     workspace_bytes, stream);
    if (rc != MOC_OK) return rc;
  }
  if (dx == nullptr && dw_qkv == nullptr) return MOC_OK;
  // do = go W_out
  rc = moc_gemm_ws(MOC_BF16, t, d, d, go, d, 1, wo, d, 1, 0, nullptr, 0, 0, nullptr, 0, 0, dox, d, MOC_BF16,
                   workspace, workspace_bytes, stream);
  if (rc == MOC_OK)
    rc = moc_rope_attention_backward_bf16(batch, seq, heads, head_dim, qkv, 3 * d, cos, sin, gdt, scale, o, lse, dox,
                                          reinterpret_cast<float*>(s + a.delta), dqkv, stream);
  // dW_qkv = dqkv^T xn, dxn = dqkv W_qkv (in do's place)
  if (rc == MOC_OK && dw_qkv != nullptr)
    rc = moc_gemm_ws(MOC_BF16, 3 * d, d, t, dqkv, 1, 3 * d, xn, d, 1, 0, nullptr, 0, 0, nullptr, 0, 0, dw_qkv, d, gdt,
                     workspace, workspace_bytes, stream);
  if (rc != MOC_OK || dx == nullptr) return rc;
  rc = moc_gemm_ws(MOC_BF16, t, d, 3 * d, dqkv, 3 * d, 1, wq, d, 1, 0, nullptr, 0, 0, nullptr, 0, 0, dox, d,
                   MOC_BF16, workspace, workspace_bytes, stream);
  if (rc != MOC_OK) return rc;
  void* part = s + a.rms;
  const int64_t pbytes = a.scratch - a.rms;
  if (f32)
    return moc_rmsnorm_backward_f32(static_cast<const float*>(x), d, t, d, static_cast<const float*>(norm_w), rstd,
                                    dox, d, static_cast<const float*>(dh), d, static_cast<float*>(dx), d,
                                    static_cast<float*>(dnorm_w), part, pbytes, stream);
  return moc_rmsnorm_backward_bf16(x, d, t, d, norm_w, rstd, dox, d, dh, d, dx, d, dnorm_w, MOC_BF16, part, pbytes,
                                   stream);
}

// ---------------------------------------------------------------------------
// The FFN half over an f32 stream with f32 weights under bf16 autocast, one
// call per pass: the weights' casts (and the incoming gradient's) in one
// launch, the norm writing the FFN's bf16 input, the FFN's launches, the
// residual sum in f32.  cast: bf16 W_gate, W_up [inter, d], W_down [d, inter]
// and, in the backward, the gradient [rows, d], one after the other, each
// 256-byte aligned.
namespace {
struct CastF32 {
  int64_t wg, wu, wd, go, bytes;
};
CastF32 cast_f32(int64_t rows, int64_t d, int64_t inter) {
  auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
  CastF32 c;
  c.wg = 0;
  c.wu = up(inter * d * 2);
  c.wd = 2 * c.wu;
  c.go = 3 * c.wu;
  c.bytes = c.go + up(rows * d * 2);
  return c;
}
}  // namespace

extern "C" int64_t moc_ffn_block_f32_cast_size(int64_t rows, int64_t d, int64_t inter) {
  return rows > 0 && d > 0 && inter > 0 ? cast_f32(rows, d, inter).bytes : 0;
}

extern "C" int moc_ffn_block_forward_f32(int64_t rows, int64_t d, int64_t inter, int64_t k, int selection,
                                         const float* h, const float* norm_w, float eps, void* xn, float* rstd,
                                         const float* wg, const float* wu, const float* wd, void* cast,
                                         int64_t cast_bytes, void* g, void* u, int64_t ld_gu, void* vals, void* idx,
                                         int idx_dtype, void* u_s, void* s_s, void* z_s, float* out, void* workspace,
                                         int64_t workspace_bytes, void* stream) {
  MOC_REQUIRE(rows >= 1 && d >= 8 && d % 8 == 0 && inter >= 8 && inter % 8 == 0, "moc_ffn_block_forward_f32: bad shape");
  MOC_REQUIRE(h && norm_w && xn && rstd && wg && wu && wd && cast && out && moc::aligned16(cast) && moc::aligned16(h) &&
                  moc::aligned16(out),
              "moc_ffn_block_forward_f32: null or unaligned operand");
  const CastF32 c = cast_f32(rows, d, inter);
  MOC_REQUIRE(cast_bytes >= c.bytes, "moc_ffn_block_forward_f32: cast buffer of %lld bytes required",
              (long long)c.bytes);
  char* b = static_cast<char*>(cast);
  const void* src[3] = {wg, wu, wd};
  void* dst[3] = {b + c.wg, b + c.wu, b + c.wd};
  const int64_t r[3] = {inter, inter, d}, cols[3] = {d, d, inter};
  int rc = moc_cast_bf16_multi(3, src, r, cols, dst, cols, stream);
  if (rc == MOC_OK) rc = moc_rmsnorm_rows_f32(h, d, rows, d, norm_w, eps, xn, d, rstd, stream);
  if (rc != MOC_OK) return rc;
  void* y = b + c.go;  // the FFN's bf16 output
  rc = ffn_forward(MOC_BF16, "moc_ffn_block_forward_f32", rows, d, inter, k, selection, xn, d, dst[0], d, dst[1], d,
                   dst[2], inter, g, u, ld_gu, vals, idx, idx_dtype, u_s, s_s, z_s, y, d, workspace, workspace_bytes,
                   stream);
  if (rc != MOC_OK) return rc;
  return moc::add_f32_bf16(h, y, out, rows * d, moc::as_stream(stream));
}

extern "C" int moc_ffn_block_backward_f32(int64_t rows, int64_t d, int64_t inter, int64_t k, const float* dout,
                                          const float* h, const float* norm_w, const float* rstd, const void* xn,
                                          const void* idx, int idx_dtype, const void* g_s, const void* u_s,
                                          const void* s_s, const void* z_s, const float* wg, const float* wu,
                                          const float* wd, void* cast, int64_t cast_bytes, void* zbuf, int64_t ldz,
                                          void* gg, void* gu, int64_t ld_ggu, int stacked, void* dxn, float* dh,
                                          float* dwg, float* dwu, float* dwd, float* dnorm_w, void* workspace,
                                          int64_t workspace_bytes, void* stream) {
  MOC_REQUIRE(rows >= 1 && d >= 8 && d % 8 == 0 && inter >= 8 && inter % 8 == 0,
              "moc_ffn_block_backward_f32: bad shape");
  MOC_REQUIRE(dout && h && norm_w && rstd && xn && wg && wu && wd && cast && dxn && dh && dnorm_w &&
                  moc::aligned16(cast) && moc::aligned16(dout),
              "moc_ffn_block_backward_f32: null or unaligned operand");
  const CastF32 c = cast_f32(rows, d, inter);
  const int64_t need = moc_ffn_block_backward_workspace_size(rows, d, inter, ld_ggu, stacked);
  MOC_REQUIRE(cast_bytes >= c.bytes && workspace != nullptr && workspace_bytes >= need && moc::aligned16(workspace),
              "moc_ffn_block_backward_f32: cast buffer of %lld and workspace of %lld bytes required",
              (long long)c.bytes, (long long)need);
  char* b = static_cast<char*>(cast);
  const void* src[4] = {wg, wu, wd, dout};
  void* dst[4] = {b + c.wg, b + c.wu, b + c.wd, b + c.go};
  const int64_t r[4] = {inter, inter, d, rows}, cols[4] = {d, d, inter, d};
  int rc = moc_cast_bf16_multi(4, src, r, cols, dst, cols, stream);
  if (rc != MOC_OK) return rc;
  const int64_t f = block_rms_offset(rows, d, inter, ld_ggu, stacked);
  rc = moc_ffn_backward_bf16(rows, d, inter, k, dst[3], d, xn, d, idx, idx_dtype, g_s, u_s, s_s, z_s, dst[0], d,
                             dst[1], d, dst[2], inter, zbuf, ldz, gg, gu, ld_ggu, stacked, nullptr, dxn, d, dwg, dwu, d,
                             dwd, inter, MOC_F32, workspace, f, stream);
  if (rc != MOC_OK) return rc;
  return moc_rmsnorm_backward_f32(h, d, rows, d, norm_w, rstd, dxn, d, dout, d, dh, d, dnorm_w,
                                  static_cast<char*>(workspace) + f, workspace_bytes - f, stream);
}

// ---------------------------------------------------------------------------
// The f32 layer's backward (moc/ffn.py:175-259, :423-497) as one call: the
// launches of the per-kernel path in its order.  s_s and z_s NULL: the GCP
// form, recomputed into s_tmp and z_tmp [rows, k].
extern "C" int64_t moc_ffn_backward_f32_workspace_size(int64_t rows, int64_t d, int64_t inter) {
  if (rows <= 0 || d <= 0 || inter <= 0) return 0;
  return std::max({gemm_ws(d, inter, rows, 0, MOC_F32), gemm_ws(rows, inter, d, 0, MOC_F32),
                   gemm_ws(inter, d, rows, 0, MOC_F32), gemm_ws(rows, d, inter, inter, MOC_F32)});
}

extern "C" int moc_ffn_backward_f32(int64_t rows, int64_t d, int64_t inter, int64_t k, const float* go,
                                    const float* x, const void* idx, int idx_dtype, const float* g_s,
                                    const float* u_s, const float* s_s, const float* z_s, float* s_tmp, float* z_tmp,
                                    const float* wg, const float* wu, const float* wd, float* zbuf, float* gg,
                                    float* gu, int64_t pitch, float* dx, float* dwg, float* dwu, float* dwd,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
  MOC_REQUIRE(rows >= 1 && d >= 4 && d % 4 == 0 && inter >= 4 && inter % 4 == 0 && k >= 1 && k <= inter &&
                  pitch >= inter && pitch % 4 == 0,
              "moc_ffn_backward_f32: bad shape");
  MOC_REQUIRE(go && x && idx && g_s && u_s && wg && wu && wd && zbuf && gg && gu && dx && dwg && dwu && dwd &&
                  (s_s != nullptr ? z_s != nullptr : (s_tmp != nullptr && z_tmp != nullptr)),
              "moc_ffn_backward_f32: null operand");
  const int64_t need = moc_ffn_backward_f32_workspace_size(rows, d, inter);
  MOC_REQUIRE(workspace_bytes >= need && (need == 0 || workspace != nullptr),
              "moc_ffn_backward_f32: workspace of %lld bytes required", (long long)need);
  int rc = MOC_OK;
  if (s_s == nullptr) {
    rc = moc_gcp_recompute(MOC_F32, g_s, u_s, rows * k, s_tmp, z_tmp, stream);
    if (rc != MOC_OK) return rc;
    s_s = s_tmp;
    z_s = z_tmp;
  }
  auto gemm = [&](int64_t m, int64_t n, int64_t kk, const float* a, int64_t am, int64_t ak, const float* b, int64_t bk,
                  float* c, int64_t ldc, const float* a2 = nullptr, const float* b2 = nullptr) {
    return moc_gemm_ws(MOC_F32, m, n, kk, a, am, ak, b, bk, 1, a2 ? kk : 0, a2, a2 ? am : 0, a2 ? ak : 0, b2,
                       b2 ? bk : 0, b2 ? 1 : 0, c, ldc, MOC_F32, workspace, workspace_bytes, stream);
  };
  rc = moc_scatter_sparse_to_dense(MOC_F32, z_s, idx, idx_dtype, rows, k, inter, zbuf, pitch, stream);
  if (rc == MOC_OK) rc = gemm(d, inter, rows, go, 1, d, zbuf, pitch, dwd, inter);  // dWd = go^T Z
  if (rc == MOC_OK) rc = gemm(rows, inter, d, go, d, 1, wd, inter, zbuf, pitch);   // gZ = go Wd, in Z's place
  if (rc == MOC_OK)
    rc = moc_sparse_backward_aux(MOC_F32, idx, idx_dtype, g_s, u_s, s_s, zbuf, pitch, rows, k, inter, gg, gu, pitch,
                                 stream);
  if (rc == MOC_OK) rc = gemm(inter, d, rows, gg, 1, pitch, x, d, dwg, d);  // dWg = gG^T x
  if (rc == MOC_OK) rc = gemm(inter, d, rows, gu, 1, pitch, x, d, dwu, d);  // dWu = gU^T x
  if (rc == MOC_OK) rc = gemm(rows, d, inter, gg, pitch, 1, wg, d, dx, d, gu, wu);  // dX = gG Wg + gU Wu
  return rc;
}
