// A run of decoder blocks launched by one call: per block the fused QKV projection with the rotary + pool write,
// the paged attention, the output projection with the residual add and norm, the SwiGLU and the down projection
// with the residual add and the next norm (model.py:99-106 in the reference), each through the entry point that
// launches it alone, with the choices a caller makes between them (a projection that splits K hands its
// partials to the kernel that follows). The results are those of the separate calls, bit for bit.
//
// A short batch's kernels take 2-17 us each, and a Python caller needs 12 us per launch, so that decode steps waited
// for the host. Launched from here: 16 rows of one token through 4 blocks (d = 2048, bf16) 440 -> 330 us, which
// are the kernels'; one row through 4 float32 blocks (d = 256) 520 -> 303; four rows of 160 tokens through
// those 707 -> 467.
#include "common.h"

namespace {

struct Shape {
  int64_t m, d, qn, qkv_n, f;   // rows, d_model, query columns, QKV columns, hidden columns
  int32_t hd, dtype;
};

// The projection's K splits are left as partials for the kernel that follows it (their sum is that kernel's).
bool partials_ok(const Shape& s, int64_t n, int64_t k) {
  return s.dtype == FS_BF16 && k % 64 == 0 && n % 8 == 0 && fs_gemm_splits(n, k, s.dtype) > 1 &&
         !fs_gemm_serial(s.m, n, k, s.dtype);
}
bool qkv_partials(const Shape& s) { return partials_ok(s, s.qkv_n, s.d) && s.hd % 16 == 0; }
bool norm_partials(const Shape& s, int64_t k) { return s.d <= 8192 && partials_ok(s, s.d, k); }
bool fused_swiglu(const Shape& s) {
  return s.dtype == FS_BF16 && s.f % 2 == 0 && s.d % 64 == 0 && fs_gemm_splits(2 * s.f, s.d, s.dtype) == 1;
}

int64_t elem_size(int32_t dtype) { return dtype == FS_F32 ? 4 : 2; }

// The scratch tensors of a block, one after the other (256-byte aligned); null base: sizes alone.
struct Scratch {
  char *qkv, *q, *o, *x1, *h2, *gu, *g, *x[2], *h[2];
  int64_t bytes;
  Scratch(char* base, const Shape& s) : bytes(0) {
    auto take = [&](int64_t cols) {
      char* p = base + bytes;
      bytes += (s.m * cols * elem_size(s.dtype) + 255) / 256 * 256;
      return p;
    };
    qkv = take(qkv_partials(s) ? 0 : s.qkv_n);
    q = take(s.qn);
    o = take(s.qn);
    x1 = take(s.d);
    h2 = take(s.d);
    gu = take(fused_swiglu(s) ? 0 : 2 * s.f);
    g = take(s.f);
    for (int i = 0; i < 2; ++i) {
      x[i] = take(s.d);
      h[i] = take(s.d);
    }
  }
};

int64_t partials_bytes(const Shape& s, int64_t n, int64_t k) {
  return (int64_t)fs_gemm_splits(n, k, s.dtype) * s.m * n * 4;
}

bool make_shape(Shape& s, int32_t B, int32_t T, int32_t n_heads, int32_t n_kv_heads, int32_t head_dim, int64_t d_model,
                int64_t ffn, int32_t dtype) {
  if (B < 0 || T < 0 || n_heads <= 0 || n_kv_heads <= 0 || head_dim <= 0 || d_model <= 0 || ffn <= 0) return false;
  if (dtype != FS_F32 && dtype != FS_BF16 && dtype != FS_F16) return false;
  s = Shape{(int64_t)B * T, d_model, (int64_t)n_heads * head_dim, (int64_t)(n_heads + 2 * n_kv_heads) * head_dim, ffn,
            head_dim, dtype};
  return true;
}

#define FS_TRY(call)          \
  do {                        \
    const int rc_ = (call);   \
    if (rc_ != 0) return rc_; \
  } while (0)

}  // namespace

extern "C" int fs_run_blocks_workspace(int32_t B, int32_t T, int32_t n_heads, int32_t n_kv_heads, int32_t head_dim,
                                       int64_t d_model, int64_t ffn, int32_t dtype, int32_t max_blocks,
                                       int32_t block_size, int64_t* bytes) {
  Shape s;
  FS_CHECK_ARG(bytes && make_shape(s, B, T, n_heads, n_kv_heads, head_dim, d_model, ffn, dtype), "run_blocks_workspace: shapes");
  int64_t g = 0;
  auto need = [&](bool partials, int64_t n, int64_t k) {
    const int64_t b = partials ? partials_bytes(s, n, k) : fs_gemm_workspace_size(s.m, n, k, dtype);
    if (b > g) g = b;
  };
  need(qkv_partials(s), s.qkv_n, s.d);
  need(norm_partials(s, s.qn), s.d, s.qn);
  need(norm_partials(s, s.f), s.d, s.f);
  need(false, s.d, s.f);   // (a last block without a norm behind it)
  if (!fused_swiglu(s)) need(false, 2 * s.f, s.d);
  bytes[0] = g;
  bytes[1] = fs_paged_attention_workspace_size(B, T, n_heads, head_dim, max_blocks, block_size);
  bytes[2] = Scratch(nullptr, s).bytes;
  return 0;
}

extern "C" int fs_run_blocks(const fs_block* blocks, int32_t n_blocks, int32_t B, int32_t T, int32_t n_heads,
                             int64_t d_model, int64_t ffn, int32_t dtype, const int32_t* positions,
                             const float* rope_cos, const float* rope_sin, int32_t rope_len, float scale, const void* x,
                             const void* h, void* x_out, void* y_out, void* gemm_ws, int64_t gemm_ws_bytes,
                             void* attn_ws, int64_t attn_ws_bytes, void* scratch, int64_t scratch_bytes, void* stream) {
  FS_CHECK_ARG(blocks && n_blocks > 0 && x && h && x_out && scratch, "run_blocks: null pointer");
  Shape s;
  FS_CHECK_ARG(make_shape(s, B, T, n_heads, blocks[0].kv.n_kv_heads, blocks[0].kv.head_dim, d_model, ffn, dtype),
               "run_blocks: shapes");
  FS_CHECK_ARG(positions && rope_cos && rope_sin && attn_ws, "run_blocks: null pointer");
  for (int32_t i = 0; i < n_blocks; ++i) {   // all of them before the first launch writes to a cache
    const fs_block& b = blocks[i];
    FS_CHECK_ARG(b.kv.n_kv_heads == blocks[0].kv.n_kv_heads && b.kv.head_dim == s.hd && b.kv.dtype == dtype,
                 "run_blocks: block %d: its cache's heads, head_dim or dtype", (int)i);
    FS_CHECK_ARG(b.w_qkv && b.w_o && b.w_gate_up && b.w_down && b.mlp_norm && b.kv.k && b.kv.v && b.tables && b.visible &&
                     (b.next_norm || i == n_blocks - 1),
                 "run_blocks: block %d: null pointer", (int)i);
  }
  FS_CHECK_ARG(blocks[n_blocks - 1].next_norm == nullptr || y_out, "run_blocks: null y_out");
  const Scratch sc(reinterpret_cast<char*>(scratch), s);
  FS_CHECK_ARG(scratch_bytes >= sc.bytes, "run_blocks: scratch %lld < %lld bytes", (long long)scratch_bytes,
               (long long)sc.bytes);
  float* parts = reinterpret_cast<float*>(gemm_ws);
  // x_to = a @ w^T + residual and, with a norm, y_to = norm(x_to)
  auto project = [&](const void* a, const void* w, int64_t k, const void* residual, const void* norm, float eps, void* x_to,
                     void* y_to) -> int {
    if (norm && norm_partials(s, k)) {
      FS_TRY(fs_gemm_partials(a, k, w, k, s.m, s.d, k, dtype, parts, gemm_ws_bytes, stream));
      return fs_splitk_add_rmsnorm(parts, fs_gemm_splits(s.d, k, dtype), residual, s.d, x_to, s.d, norm, y_to, s.d, s.m,
                                   s.d, eps, dtype, stream);
    }
    FS_TRY(fs_gemm(a, k, w, k, x_to, s.d, residual, s.d, s.m, s.d, k, dtype, gemm_ws, gemm_ws_bytes, stream));
    if (!norm) return 0;
    return fs_add_rmsnorm(x_to, s.d, nullptr, 0, nullptr, 0, norm, y_to, s.d, s.m, s.d, eps, dtype, stream);
  };
  for (int32_t i = 0; i < n_blocks; ++i) {
    const fs_block& b = blocks[i];
    if (qkv_partials(s)) {
      FS_TRY(fs_gemm_partials(h, s.d, b.w_qkv, s.d, s.m, s.qkv_n, s.d, dtype, parts, gemm_ws_bytes, stream));
      FS_TRY(fs_qkv_rope_write_partials(parts, fs_gemm_splits(s.qkv_n, s.d, dtype), s.m, s.qkv_n, T, n_heads, positions,
                                        b.slots, rope_cos, rope_sin, rope_len, b.tables, b.table_stride, b.max_blocks,
                                        &b.kv, sc.q, s.qn, stream));
    } else {
      FS_TRY(fs_gemm(h, s.d, b.w_qkv, s.d, sc.qkv, s.qkv_n, nullptr, 0, s.m, s.qkv_n, s.d, dtype, gemm_ws, gemm_ws_bytes,
                     stream));
      FS_TRY(fs_qkv_rope_write(sc.qkv, s.qkv_n, s.m, T, n_heads, positions, b.slots, rope_cos, rope_sin, rope_len,
                               b.tables, b.table_stride, b.max_blocks, &b.kv, sc.q, s.qn, stream));
    }
    auto attend = b.reuse_plan ? fs_paged_attention_reuse_plan : fs_paged_attention;
    FS_TRY(attend(sc.q, T * s.qn, s.qn, s.hd, &b.kv, b.tables, b.table_stride, b.max_blocks, b.visible, B, T, n_heads,
                  scale, sc.o, T * s.qn, s.qn, s.hd, attn_ws, attn_ws_bytes, stream));
    FS_TRY(project(sc.o, b.w_o, s.qn, x, b.mlp_norm, b.mlp_eps, sc.x1, sc.h2));
    if (fused_swiglu(s)) {
      FS_TRY(fs_gemm_swiglu(sc.h2, s.d, b.w_gate_up, s.d, sc.g, s.f, s.m, s.f, s.d, dtype, stream));
    } else {
      FS_TRY(fs_gemm(sc.h2, s.d, b.w_gate_up, s.d, sc.gu, 2 * s.f, nullptr, 0, s.m, 2 * s.f, s.d, dtype, gemm_ws,
                     gemm_ws_bytes, stream));
      FS_TRY(fs_silu_mul(sc.gu, 2 * s.f, sc.g, s.f, s.m, s.f, dtype, stream));
    }
    const bool last = i == n_blocks - 1;
    void* xn = last ? x_out : sc.x[i & 1];
    void* hn = last ? y_out : sc.h[i & 1];
    FS_TRY(project(sc.g, b.w_down, s.f, sc.x1, b.next_norm, b.next_eps, xn, hn));
    x = xn;
    h = hn;
  }
  return 0;
}
