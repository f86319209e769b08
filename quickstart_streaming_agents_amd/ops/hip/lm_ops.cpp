// Torch bindings of the decoder-mixer kernels (module qsa_lm_hip).  Every
// binding checks shapes, types and strides against what its kernel and grid
// assume; the matrix-core variants are chosen here where the sizes fit them.
#include <hip/hip_runtime.h>
#include <torch/extension.h>
#include <ATen/TracerMode.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/HIPContext.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include "step_args.h"

#define CHK_DEV(t) TORCH_CHECK((t).is_cuda(), #t " must be on the GPU")
#define CHK_CONT(t) TORCH_CHECK((t).is_contiguous(), #t " must be contiguous")
#define CHK_F32(t) TORCH_CHECK((t).scalar_type() == at::kFloat && (t).is_contiguous(), #t " must be contiguous f32")
#define CHK_I32(t) TORCH_CHECK((t).scalar_type() == at::kInt && (t).is_contiguous(), #t " must be contiguous i32")
#define CHK_SAME(a, b) TORCH_CHECK((a).scalar_type() == (b).scalar_type(), #a " and " #b " must have one dtype")

using torch::Tensor;
using OptTensor = c10::optional<Tensor>;

static inline hipStream_t cur_stream() {
  return at::hip::getCurrentHIPStream().stream();
}
static inline int is_f32(const Tensor& t) {
  TORCH_CHECK(t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16,
              "bf16 or f32 expected");
  return t.scalar_type() == at::kFloat;
}
static inline bool aligned(const Tensor& t, int bytes) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % bytes == 0;
}
static inline void chk_rows(const Tensor& t, const char* name) {
  TORCH_CHECK(t.dim() == 2 && t.stride(1) == 1, name,
              " must be 2-D with contiguous rows");
}
// a kernel given a host tensor's pointer would read the host's memory
template <typename... Ts>
static inline void chk_there(const Tensor& like, const Ts&... t) {
  TORCH_CHECK(((t.device() == like.device()) && ...), "operands must be on ",
              like.device());
}
static inline const bf16_t* u16(const Tensor& t) {
  return reinterpret_cast<const bf16_t*>(t.data_ptr());
}
static inline bf16_t* u16m(const Tensor& t) {
  return reinterpret_cast<bf16_t*>(t.data_ptr());
}

extern "C" void qsa_residual_norm_launch(float*, const void*, long long,
    const float*, int, const void*, const void*, const long long*, float, const void*,
    const void*, const void*, void*, long long, int, int, float, int, int,
    int, int, hipStream_t);
extern "C" void qsa_rmsnorm_launch(const bf16_t*, const bf16_t*, bf16_t*, bf16_t*,
    long long, int, float, hipStream_t);
extern "C" void qsa_short_gemm_launch(const bf16_t*, const bf16_t*, bf16_t*, int, int,
    int, long long, int, hipStream_t);
extern "C" bool qsa_short_gemm_takes(long long, long long, long long);
extern "C" void qsa_encoder_attn_launch(const bf16_t*, const float*, const float*, int,
    const int*, const int*, const int*, const int*, bf16_t*, int, int, int, float,
    hipStream_t);
extern "C" void qsa_rmsnorm_shares_launch(const float*, int, bf16_t*,
    const bf16_t*, bf16_t*, long long, int, float, hipStream_t);
extern "C" void qsa_glu_launch(const void*, const float*, int, const void*,
    const long long*,
    void*, long long, long long, long long, long long, long long, int, int,
    int, hipStream_t);
extern "C" void qsa_conv_qkv_launch(ConvQkv, long long, int, int, int, hipStream_t);
extern "C" void qsa_conv_silu_launch(const void*, long long, const float*,
    const float*, int, void*, ConvStep, long long, int, void*, int, int, int,
    hipStream_t);
extern "C" void qsa_gqa_rows_launch(const void*, const void*, const void*,
    const int*, int, const int*, const int*, const float*, const void*,
    long long, void*, long long, int, int, int, int, int, float, float, int,
    hipStream_t);
extern "C" void qsa_gqa_rows_mfma_launch(const bf16_t*, const bf16_t*,
    const bf16_t*, const int*, int, const int*, const int*, const float*,
    const bf16_t*, long long, float*, float*, bf16_t*, long long, int, int,
    int, int, int, float, float, int, hipStream_t);
extern "C" void qsa_gqa_portions_launch(const bf16_t*, const bf16_t*,
    const bf16_t*, const int*, int, const float*, const bf16_t*, long long,
    const int*, const int*, const int*, const int*, const int*, bf16_t*,
    long long, int, int, int, int, int, float, float, int, hipStream_t);
extern "C" void qsa_ssd_decode_launch(const void*, long long, int, int,
    const void*, const float*, const float*, const float*, float*, const int*,
    const int*, void*, int, int, int, int, int, int, int, hipStream_t);
extern "C" int qsa_ssd_step_rows(int, int, int, int, int, int);
extern "C" void qsa_ssd_step_launch(SsdStep, hipStream_t);
extern "C" void qsa_ssd_seq_launch(const void*, long long, int, int,
    const void*, const float*, const float*, const float*, float*, const int*,
    const int*, const int*, const int*, void*, int, int, int, int, int, int,
    hipStream_t);
extern "C" void qsa_ssd_steps_launch(const bf16_t*, long long, int,
    const float*, const float*, const int*, const int*, const int*,
    const int*, float*, int, int, hipStream_t);
extern "C" void qsa_ssd_state_launch(const bf16_t*, const float*, float*,
    const int*, const int*, const int*, const int*, const int*, void*, int,
    int, int, int, int, int, int, hipStream_t);
extern "C" void qsa_ssd_out_launch(const bf16_t*, long long, int,
    const bf16_t*, const float*, const float*, const int*, const int*,
    const int*, const int*, const int*, const void*, int, bf16_t*, int, int,
    int, int, int, int, hipStream_t);
extern "C" void qsa_part_norm_launch(const void*, const float*, void*,
    long long, long long, int, int, float, int, int, hipStream_t);
extern "C" void qsa_latent_norm_store_launch(const void*, long long,
    const void*, const void*, void*, void*, const int*, long long, int, int,
    float, int, hipStream_t);
extern "C" void qsa_decode_slots_launch(const int*, const int*, int*, int,
    int, hipStream_t);
extern "C" void qsa_argmax_rows_launch(const void*, long long*, long long,
    int, int, hipStream_t);
extern "C" void qsa_retention_decode_launch(const void*, long long,
    const float*, const float*, const float*, float*, const int*, const int*,
    void*, int, int, int, int, int, float, float, int, int, int, hipStream_t);
extern "C" void qsa_retention_seq_launch(const void*, long long,
    const float*, const float*, const float*, float*, const int*, const int*,
    const int*, const int*, void*, int, int, int, int, int, float, float,
    int, int, hipStream_t);
extern "C" void qsa_retention_rotate_launch(const bf16_t*, long long,
    const float*, const float*, const int*, bf16_t*, long long, int, int,
    int, int, float, int, hipStream_t);
extern "C" void qsa_retention_state_launch(const bf16_t*, long long,
    long long, const bf16_t*, long long, const float*, float*, const int*,
    const int*, const int*, const int*, const int*, void*, int, int, int,
    int, int, int, hipStream_t);
extern "C" void qsa_retention_out_launch(const bf16_t*, long long, long long,
    const bf16_t*, long long, const float*, const int*, const int*,
    const int*, const int*, const int*, const void*, long long, bf16_t*,
    int, int, int, int, float, hipStream_t);
extern "C" void qsa_head_matmul_launch(const void*, long long, const void*,
    const void*, long long, void*, int, int, int, int, int, int, hipStream_t);
extern "C" void qsa_latent_rows_launch(const void*, const void*, const int*,
    int, const int*, const int*, const void*, void*, int, int, int, int,
    float, int, hipStream_t);
extern "C" void qsa_latent_rows_mfma_launch(const bf16_t*, const bf16_t*,
    const int*, int, const int*, const int*, const bf16_t*, float*, float*,
    bf16_t*, int, int, int, int, float, int, hipStream_t);
extern "C" void qsa_window_attn_prefill_launch(const bf16_t*, long long,
    const bf16_t*, long long, const bf16_t*, long long, const bf16_t*,
    const int*, const int*, const int*, const int*, const int*, const int*,
    const int*, bf16_t*, int, int, int, int, int, float, hipStream_t);
extern "C" void qsa_skinny_gemm_launch(const bf16_t*, const bf16_t*, bf16_t*,
    int, int, long long, long long, bool, hipStream_t);
extern "C" int qsa_rows_gemm_plan(int, int, int, int, int, int*, float*);
extern "C" bool qsa_wide_gemm_fits(int, int, int);
extern "C" float qsa_wide_gemm_plan(int, int, int, int, int*, int*, int*);
extern "C" void qsa_wide_gemm_launch(const bf16_t*, const bf16_t*, bf16_t*, int,
                                     int, int, long long, int, int, hipStream_t);
extern "C" void qsa_rows_gemm_launch(const bf16_t*, const bf16_t*, bf16_t*,
    float*, int, int, int, long long, int, int, int, bool, hipStream_t);

// Whether t [S, rows, cols] is a product of bf16 rows whose shares of K have not
// been added (gemm_parts)
static bool is_shares(const Tensor& t, const Tensor& like, int64_t rows,
                      int64_t cols) {
  if (t.dim() != 3) return false;
  TORCH_CHECK(t.scalar_type() == at::kFloat && t.is_contiguous() &&
                  t.device() == like.device() && t.size(0) >= 1 &&
                  t.size(1) == rows && t.size(2) == cols && cols % 8 == 0 &&
                  like.scalar_type() == at::kBFloat16 && aligned(t, 16),
              "shares [S, rows, cols], f32, of bf16 rows");
  return true;
}

static Tensor add_shares(const Tensor& parts) {
  Tensor sum = parts[0];
  for (int64_t s = 1; s < parts.size(0); ++s) sum = sum + parts[s];
  return sum.to(at::kBFloat16);
}

// res [T, W] f32 updated in place; returns norm(res) * w (+ b), or res itself
// in y's storage type when w is not given
Tensor residual_norm(Tensor res, OptTensor y, OptTensor table, OptTensor ids,
                     OptTensor vec, OptTensor w, OptTensor b, double eps,
                     bool init, bool layer, OptTensor post, double tscale) {
  CHK_DEV(res); CHK_F32(res);
  TORCH_CHECK(res.dim() == 2, "res [T, W]");
  TORCH_CHECK(w || y, "norm weight or y");
  const long long T = res.size(0);
  const int W = (int)res.size(1);
  const bool shares = y && y->dim() == 3;
  const auto opts = w ? w->options()
                      : y->options().dtype(shares ? at::kBFloat16
                                                  : y->scalar_type());
  auto out = torch::empty({T, (long long)W}, opts);
  const Tensor& like = out;
  const int f32 = is_f32(like);
  if (T == 0) return out;
  bool v4 = W % 4 == 0;
  const int word = f32 ? 16 : 8;
  auto row_vec = [&](const OptTensor& t, const char* name) -> const void* {
    if (!t) return nullptr;
    CHK_SAME(*t, like); CHK_CONT(*t);
    TORCH_CHECK(t->numel() == W, name, " size");
    v4 = v4 && aligned(*t, word);
    return t->data_ptr();
  };
  const void* wp = row_vec(w, "norm weight");
  const void* bp = row_vec(b, "bias");
  const void* vp = row_vec(vec, "vec");
  const void* pp = row_vec(post, "post-norm weight");
  TORCH_CHECK(!post || y, "post needs y");
  TORCH_CHECK(w || !b, "bias without weight");
  const void *yp = nullptr, *tp = nullptr;
  long long ys = 0;
  int vocab = 0;
  const long long* ip = nullptr;
  if (shares) {
    is_shares(*y, like, T, W);
  } else if (y) {
    CHK_SAME(*y, like); chk_rows(*y, "y");
    TORCH_CHECK(y->size(0) == T && y->size(1) == W, "y shape");
    yp = y->data_ptr(); ys = y->stride(0);
    v4 = v4 && ys % 4 == 0 && aligned(*y, word);
  }
  if (table) {
    TORCH_CHECK(ids.has_value(), "table needs ids");
    CHK_SAME(*table, like); CHK_CONT(*table); CHK_CONT(*ids);
    TORCH_CHECK(ids->scalar_type() == at::kLong && ids->numel() == T, "ids");
    TORCH_CHECK(table->dim() == 2 && table->size(1) == W, "table shape");
    tp = table->data_ptr(); vocab = (int)table->size(0);
    ip = reinterpret_cast<const long long*>(ids->data_ptr<int64_t>());
    v4 = v4 && aligned(*table, word);
  }
  if (shares && !v4)                   // rows that the kernel reads one by one
    return residual_norm(res, add_shares(*y), table, ids, vec, w, b, eps, init,
                         layer, post, tscale);
  qsa_residual_norm_launch(res.data_ptr<float>(), yp, ys,
                           shares ? y->data_ptr<float>() : nullptr,
                           shares ? (int)y->size(0) : 0, pp, tp, ip,
                           (float)tscale, vp, wp, bp, out.data_ptr(), T, W,
                           vocab, (float)eps, init, layer, f32, v4,
                           cur_stream());
  return out;
}

Tensor glu(Tensor gate, Tensor up, bool gelu) {
  CHK_DEV(gate); chk_rows(gate, "gate"); chk_rows(up, "up");
  CHK_SAME(gate, up);
  TORCH_CHECK(gate.sizes() == up.sizes(), "gate/up shapes must match");
  const long long rows = gate.size(0), cols = gate.size(1);
  auto out = torch::empty({rows, cols}, gate.options());
  if (rows == 0 || cols == 0) return out;
  const int v = cols % 8 == 0 && gate.stride(0) % 8 == 0 &&
                up.stride(0) % 8 == 0 && aligned(gate, 16) && aligned(up, 16);
  qsa_glu_launch(gate.data_ptr(), nullptr, 0, up.data_ptr(), nullptr,
                 out.data_ptr(),
                 rows, cols, gate.stride(0), up.stride(0), 0, gelu,
                 is_f32(gate), v, cur_stream());
  return out;
}

// act(gate [T, n]) * table[ids, col0 : col0 + n]
Tensor glu_table(Tensor gate, Tensor table, Tensor ids, long col0,
                 bool gelu) {
  CHK_DEV(gate); CHK_CONT(table); CHK_CONT(ids);
  const bool shares = gate.dim() == 3;
  const long long rows = gate.size(shares ? 1 : 0);
  const long long cols = gate.size(shares ? 2 : 1);
  if (shares) {
    is_shares(gate, table, rows, cols);
  } else {
    chk_rows(gate, "gate"); CHK_SAME(gate, table);
  }
  TORCH_CHECK(ids.scalar_type() == at::kLong && ids.numel() == rows, "ids");
  TORCH_CHECK(table.dim() == 2 && col0 >= 0 && table.size(0) > 0 &&
                  col0 + cols <= table.size(1), "columns of the table");
  auto out = torch::empty({rows, cols}, table.options());
  if (rows == 0 || cols == 0) return out;
  const int v = cols % 8 == 0 && (shares || gate.stride(0) % 8 == 0) &&
                col0 % 8 == 0 && table.size(1) % 8 == 0 && aligned(gate, 16) &&
                aligned(table, 16);
  if (shares && !v)
    return glu_table(add_shares(gate), table, ids, col0, gelu);
  const char* base = reinterpret_cast<const char*>(table.data_ptr()) +
                     col0 * table.element_size();
  qsa_glu_launch(shares ? nullptr : gate.data_ptr(),
                 shares ? gate.data_ptr<float>() : nullptr,
                 shares ? (int)gate.size(0) : 0, base,
                 reinterpret_cast<const long long*>(ids.data_ptr<int64_t>()),
                 out.data_ptr(), rows, cols, shares ? 0 : gate.stride(0),
                 table.size(1), table.size(0), gelu, is_f32(table), v,
                 cur_stream());
  return out;
}

// x [T, >= qr+kr]; returns rms(x[:, :qr]) * wq; the latent goes to the cache
Tensor latent_norm_store(Tensor x, Tensor wq, Tensor wk, Tensor cache,
                         Tensor slots, double eps) {
  CHK_DEV(x); chk_rows(x, "x"); CHK_CONT(wq); CHK_CONT(wk); CHK_CONT(cache);
  CHK_SAME(x, wq); CHK_SAME(x, wk); CHK_SAME(x, cache); CHK_I32(slots);
  const long long T = x.size(0);
  const int qr = (int)wq.numel(), kr = (int)wk.numel();
  TORCH_CHECK(x.size(1) >= qr + kr, "x holds [q latent | kv latent]");
  TORCH_CHECK(cache.dim() == 3 && cache.size(1) == 64 && cache.size(2) == kr,
              "latent cache [pages, 64, kr]");
  TORCH_CHECK(slots.numel() == T, "one slot per row");
  auto cq = torch::empty({T, (long long)qr}, x.options());
  if (T == 0) return cq;
  qsa_latent_norm_store_launch(x.data_ptr(), x.stride(0), wq.data_ptr(),
                               wk.data_ptr(), cq.data_ptr(),
                               cache.data_ptr(), slots.data_ptr<int>(), T, qr,
                               kr, (float)eps, is_f32(x), cur_stream());
  return cq;
}

Tensor decode_slots(Tensor block_table, Tensor seq_lens) {
  CHK_DEV(block_table); CHK_I32(block_table); CHK_I32(seq_lens);
  const int B = (int)seq_lens.numel();
  TORCH_CHECK(block_table.dim() == 2 && block_table.size(0) == B, "table rows");
  auto slots = torch::empty({B}, seq_lens.options());
  if (B)
    qsa_decode_slots_launch(block_table.data_ptr<int>(),
                            seq_lens.data_ptr<int>(), slots.data_ptr<int>(),
                            B, (int)block_table.size(1), cur_stream());
  return slots;
}

Tensor argmax_rows(Tensor x) {
  CHK_DEV(x); CHK_CONT(x);
  TORCH_CHECK(x.dim() == 2 && x.size(1) > 0, "x [rows, n]");
  auto out = torch::empty({x.size(0)}, x.options().dtype(at::kLong));
  if (x.size(0))
    qsa_argmax_rows_launch(x.data_ptr(),
                           reinterpret_cast<long long*>(out.data_ptr<int64_t>()),
                           x.size(0), (int)x.size(1), is_f32(x),
                           cur_stream());
  return out;
}

// ---- retention -------------------------------------------------------------
struct RetDims { int H, D, E, rot, table_len; };

static RetDims ret_check(const Tensor& x, const Tensor& cos_t,
                         const Tensor& sin_t, const Tensor& decay,
                         const Tensor& state, long rot) {
  CHK_DEV(x); chk_rows(x, "x"); CHK_F32(state); CHK_F32(decay);
  TORCH_CHECK(state.dim() == 4, "state [slots, H, D, E]");
  RetDims r{(int)state.size(1), (int)state.size(2), (int)state.size(3),
            (int)rot, 0x7fffffff};
  TORCH_CHECK(decay.numel() == r.H, "one decay per head");
  TORCH_CHECK(x.size(1) >= 2LL * r.H * r.D + 2LL * r.H * r.E,
              "x holds [q | k | v | gate]");
  TORCH_CHECK(rot % 2 == 0 && rot >= 0 && rot <= r.D, "rotated dims");
  if (rot > 0) {
    CHK_F32(cos_t); CHK_F32(sin_t);
    TORCH_CHECK(cos_t.dim() == 2 && cos_t.size(1) == rot / 2 &&
                    sin_t.sizes() == cos_t.sizes(), "rotation tables");
    r.table_len = (int)cos_t.size(0);
  }
  return r;
}

Tensor retention_decode(Tensor x, Tensor cos_t, Tensor sin_t, Tensor decay,
                        Tensor state, Tensor slots, Tensor seq_lens, long rot,
                        double kscale, double eps) {
  const RetDims r = ret_check(x, cos_t, sin_t, decay, state, rot);
  CHK_I32(slots); CHK_I32(seq_lens);
  const int B = (int)x.size(0);
  TORCH_CHECK(slots.numel() == B && seq_lens.numel() == B, "slots/seq_lens");
  TORCH_CHECK(2 * r.D + 2 * r.E <= 8000, "head too wide for the decode block");
  auto out = torch::empty({B, (long long)r.H * r.E}, x.options());
  if (B == 0) return out;
  if (r.D == 0 || r.E == 0) return out.zero_();   // no state to ask for
  const int v4 = r.E % 4 == 0 && (2LL * r.H * r.D) % 4 == 0 &&
                 x.stride(0) % 4 == 0 && aligned(x, 16);
  qsa_retention_decode_launch(
      x.data_ptr(), x.stride(0), cos_t.data_ptr<float>(),
      sin_t.data_ptr<float>(), decay.data_ptr<float>(),
      state.data_ptr<float>(), slots.data_ptr<int>(),
      seq_lens.data_ptr<int>(), out.data_ptr(), B, r.H, r.D, r.E, r.rot,
      (float)kscale, (float)eps, r.table_len, is_f32(x), v4, cur_stream());
  return out;
}

static int chk_items(const Tensor& slots, const Tensor& off,
                     const Tensor& start, const Tensor& len) {
  CHK_I32(slots); CHK_I32(off); CHK_I32(start); CHK_I32(len);
  const int n = (int)slots.numel();
  TORCH_CHECK(off.numel() == n && start.numel() == n && len.numel() == n,
              "per-portion arrays");
  return n;
}

// rows of x outside the portions are left unwritten in `out`
void retention_seq(Tensor x, Tensor cos_t, Tensor sin_t, Tensor decay,
                   Tensor state, Tensor slots, Tensor off, Tensor start,
                   Tensor len, Tensor out, long rot, double kscale,
                   double eps) {
  const RetDims r = ret_check(x, cos_t, sin_t, decay, state, rot);
  const int n = chk_items(slots, off, start, len);
  CHK_SAME(x, out); CHK_CONT(out);
  TORCH_CHECK(out.size(0) == x.size(0) && out.size(1) == (long long)r.H * r.E,
              "out [T, H*E]");
  TORCH_CHECK(2 * r.D + r.E <= 12000, "head too wide");
  if (n == 0) return;
  qsa_retention_seq_launch(
      x.data_ptr(), x.stride(0), cos_t.data_ptr<float>(),
      sin_t.data_ptr<float>(), decay.data_ptr<float>(),
      state.data_ptr<float>(), slots.data_ptr<int>(), off.data_ptr<int>(),
      start.data_ptr<int>(), len.data_ptr<int>(), out.data_ptr(), n, r.H, r.D,
      r.E, r.rot, (float)kscale, (float)eps, r.table_len, is_f32(x),
      cur_stream());
}

static int pad_dim(int d) {
  int p = 32;
  while (p < d) p *= 2;
  return p;
}

bool retention_chunked_ok(long H, long D, long E) {
  return D <= 256 && E <= 512 && E % 8 == 0 && (2 * H * D) % 8 == 0 &&
         (H * E) % 8 == 0;
}

// chunked prefill of the portions; rows r0.. of x are the portions' rows
void retention_chunked(Tensor x, Tensor cos_t, Tensor sin_t,
                       Tensor log2_decay, Tensor state, Tensor slots,
                       Tensor off, Tensor start, Tensor len,
                       Tensor positions, Tensor chunk0, Tensor chunk_item,
                       Tensor chunk_t0, Tensor out, long rot, double kscale,
                       double eps) {
  const RetDims r = ret_check(x, cos_t, sin_t, log2_decay, state, rot);
  const int n = chk_items(slots, off, start, len);
  CHK_SAME(x, out); CHK_CONT(out); CHK_I32(positions); CHK_I32(chunk0);
  CHK_I32(chunk_item); CHK_I32(chunk_t0);
  TORCH_CHECK(x.scalar_type() == at::kBFloat16, "bf16 storage");
  TORCH_CHECK(retention_chunked_ok(r.H, r.D, r.E), "sizes of the chunked path");
  TORCH_CHECK(x.stride(0) % 8 == 0 && aligned(x, 16), "x alignment");
  const long long T = x.size(0), nc = chunk_item.numel();
  TORCH_CHECK(positions.numel() == T && chunk0.numel() == n &&
                  chunk_t0.numel() == nc, "plan arrays");
  TORCH_CHECK(out.size(0) == T && out.size(1) == (long long)r.H * r.E, "out");
  if (n == 0 || nc == 0) return;
  const int DP = pad_dim(r.D), EP = (r.E + 15) / 16 * 16;
  auto planes = torch::empty({4, T, r.H, DP}, x.options());
  auto prefix = torch::empty({nc, r.H, 2, EP, DP}, x.options());
  hipStream_t st = cur_stream();
  const long long voff = 2LL * r.H * r.D;
  qsa_retention_rotate_launch(u16(x), x.stride(0), cos_t.data_ptr<float>(),
                              sin_t.data_ptr<float>(),
                              positions.data_ptr<int>(), u16m(planes), T, r.H,
                              r.D, DP, r.rot, (float)kscale, r.table_len, st);
  qsa_retention_state_launch(u16(x), x.stride(0), voff, u16(planes), T,
                             log2_decay.data_ptr<float>(),
                             state.data_ptr<float>(), slots.data_ptr<int>(),
                             off.data_ptr<int>(), start.data_ptr<int>(),
                             len.data_ptr<int>(), chunk0.data_ptr<int>(),
                             prefix.data_ptr(), n, r.H, r.D, DP, r.E, EP, st);
  qsa_retention_out_launch(u16(x), x.stride(0), voff, u16(planes), T,
                           log2_decay.data_ptr<float>(), off.data_ptr<int>(),
                           start.data_ptr<int>(), len.data_ptr<int>(),
                           chunk_item.data_ptr<int>(),
                           chunk_t0.data_ptr<int>(), prefix.data_ptr(), nc,
                           u16m(out), r.H, DP, r.E, EP, (float)eps, st);
}

// ---- latent attention ------------------------------------------------------
// x [M, H, K] rows (row stride free), W [H, N, K] -> [M, H*N]
Tensor head_matmul(Tensor x, Tensor W, OptTensor gate) {
  CHK_DEV(x); chk_rows(x, "x"); CHK_CONT(W); CHK_SAME(x, W);
  TORCH_CHECK(W.dim() == 3, "W [H, N, K]");
  const int H = (int)W.size(0), N = (int)W.size(1), K = (int)W.size(2);
  TORCH_CHECK(x.size(1) == (long long)H * K, "x [M, H*K]");
  TORCH_CHECK(K <= 16000, "K");
  const int M = (int)x.size(0);
  auto out = torch::empty({M, (long long)H * N}, x.options());
  if (M == 0) return out;
  const int f32 = is_f32(x);
  int mfma = !f32 && K % 8 == 0 && N % 4 == 0 && x.stride(0) % 8 == 0 &&
             aligned(x, 16) && aligned(W, 16);
  const void* gp = nullptr;
  long long gs = 0;
  if (gate) {
    CHK_SAME(x, *gate); chk_rows(*gate, "gate");
    TORCH_CHECK(gate->size(0) == M && gate->size(1) == (long long)H * N,
                "gate [M, H*N]");
    gp = gate->data_ptr(); gs = gate->stride(0);
    mfma = mfma && gs % 4 == 0 && aligned(*gate, 8);
  }
  qsa_head_matmul_launch(x.data_ptr(), x.stride(0), W.data_ptr(), gp, gs,
                         out.data_ptr(), M, H, N, K, f32, mfma, cur_stream());
  return out;
}

// qa [R, H*KR] absorbed queries -> normalized latent read-out [R, H*KR].
// row_item: which block_table row a query row uses (none: its own index);
// row_len: position + 1 of the query row (0: row not in use).
Tensor latent_rows(Tensor qa, Tensor cache, Tensor block_table,
                   OptTensor row_item, Tensor row_len, Tensor sink,
                   long window, double scale) {
  CHK_DEV(qa); CHK_CONT(qa); CHK_CONT(cache); CHK_SAME(qa, cache);
  CHK_SAME(qa, sink); CHK_CONT(sink); CHK_I32(block_table); CHK_I32(row_len);
  const int R = (int)qa.size(0), H = (int)sink.numel();
  TORCH_CHECK(cache.dim() == 3 && cache.size(1) == 64, "cache [P, 64, KR]");
  const int KR = (int)cache.size(2);
  TORCH_CHECK(qa.dim() == 2 && qa.size(1) == (long long)H * KR, "qa [R, H*KR]");
  TORCH_CHECK(row_len.numel() == R && block_table.dim() == 2, "row arrays");
  TORCH_CHECK(KR <= 8000, "latent too wide");
  const int* ri = nullptr;
  if (row_item) {
    CHK_I32(*row_item);
    TORCH_CHECK(row_item->numel() == R, "row_item");
    ri = row_item->data_ptr<int>();
  } else {
    TORCH_CHECK(block_table.size(0) >= R, "block_table rows");
  }
  auto out = torch::empty_like(qa);
  if (R == 0) return out;
  const int mp = (int)block_table.size(1);
  const int f32 = is_f32(qa);
  if (!f32 && KR % 8 == 0 && KR <= 512) {
    const int HT = (H + 15) / 16;
    int pages = mp;
    if (window > 0) pages = (int)std::min<long>(mp, (window + 62) / 64 + 1);
    // two blocks fit a CU: enough of them to fill the chip once, and no
    // shares that differ by a page when they need not
    long long ns = (512 + (long long)R * HT - 1) / ((long long)R * HT);
    ns = std::max<long long>(1, std::min<long long>(ns, pages));
    const long long per = (pages + ns - 1) / ns;
    ns = (pages + per - 1) / per;
    auto of = qa.options().dtype(at::kFloat);
    auto po = torch::empty({R, H, ns, KR}, of);
    auto pm = torch::empty({R, H, ns, 2}, of);
    qsa_latent_rows_mfma_launch(
        u16(qa), u16(cache), block_table.data_ptr<int>(), mp, ri,
        row_len.data_ptr<int>(), u16(sink), po.data_ptr<float>(),
        pm.data_ptr<float>(), u16m(out), R, H, KR, (int)window, (float)scale,
        (int)ns, cur_stream());
  } else {
    qsa_latent_rows_launch(qa.data_ptr(), cache.data_ptr(),
                           block_table.data_ptr<int>(), mp, ri,
                           row_len.data_ptr<int>(), sink.data_ptr(),
                           out.data_ptr(), R, H, KR, (int)window,
                           (float)scale, f32, cur_stream());
  }
  return out;
}

bool window_attn_ok(long H, long D, long E) {
  return D <= 256 && E <= 256 && D % 8 == 0 && E % 8 == 0;
}

// portions' rows of q [T, H*D] against expanded context kv [C, H*(D+E)];
// writes sigmoid(gate) * attention into the same rows of out [T, H*E]
void window_attn_prefill(Tensor q, Tensor kv, Tensor gate, Tensor sink,
                         Tensor qb_item, Tensor qb_t0, Tensor off,
                         Tensor start, Tensor len, Tensor ctx_off,
                         Tensor ctx_pos, Tensor out, long D, long E,
                         long window, double scale) {
  CHK_DEV(q); chk_rows(q, "q"); chk_rows(kv, "kv"); chk_rows(gate, "gate");
  CHK_CONT(out); CHK_CONT(sink);
  TORCH_CHECK(q.scalar_type() == at::kBFloat16, "bf16 storage");
  CHK_SAME(q, kv); CHK_SAME(q, gate); CHK_SAME(q, sink); CHK_SAME(q, out);
  CHK_I32(qb_item); CHK_I32(qb_t0); CHK_I32(off); CHK_I32(start);
  CHK_I32(len); CHK_I32(ctx_off); CHK_I32(ctx_pos);
  const int H = (int)sink.numel();
  TORCH_CHECK(window_attn_ok(H, D, E), "head sizes of the matrix-core path");
  TORCH_CHECK(q.size(1) == H * D && kv.size(1) == H * (D + E) &&
                  gate.size(1) == H * E && out.size(1) == H * E &&
                  gate.size(0) == q.size(0) && out.size(0) == q.size(0),
              "operand shapes");
  TORCH_CHECK(q.stride(0) % 8 == 0 && kv.stride(0) % 8 == 0 &&
                  gate.stride(0) % 4 == 0 && aligned(q, 16) &&
                  aligned(kv, 16) && aligned(gate, 8), "alignment");
  const int QB = (int)qb_item.numel();
  const auto n = off.numel();
  TORCH_CHECK(qb_t0.numel() == QB && start.numel() == n && len.numel() == n &&
                  ctx_off.numel() == n && ctx_pos.numel() == n, "plan arrays");
  if (QB == 0) return;
  qsa_window_attn_prefill_launch(
      u16(q), q.stride(0), u16(kv), kv.stride(0), u16(gate), gate.stride(0),
      u16(sink), qb_item.data_ptr<int>(), qb_t0.data_ptr<int>(),
      off.data_ptr<int>(), start.data_ptr<int>(), len.data_ptr<int>(),
      ctx_off.data_ptr<int>(), ctx_pos.data_ptr<int>(), u16m(out), QB, H,
      (int)D, (int)E, (int)window, (float)scale, cur_stream());
}

// ---- short convolutions ----------------------------------------------------
// Portions with chunks of 16 rows (item, t0), or, without `item`, one token
// per row at position start - 1.
static int conv_step(ConvStep& st, const OptTensor& item, const OptTensor& t0,
                     const OptTensor& off, const Tensor& start,
                     const OptTensor& len, const Tensor& slots, long rows) {
  CHK_I32(start); CHK_I32(slots);
  TORCH_CHECK(start.numel() == slots.numel(), "one slot per portion");
  st = ConvStep{nullptr, nullptr, nullptr, start.data_ptr<int>(), nullptr,
                slots.data_ptr<int>()};
  if (!item) {
    TORCH_CHECK(start.numel() == rows, "one row per sequence");
    return (int)rows;
  }
  TORCH_CHECK(t0 && off && len, "portions need t0, off and len");
  CHK_I32(*item); CHK_I32(*t0); CHK_I32(*off); CHK_I32(*len);
  TORCH_CHECK(t0->numel() == item->numel() &&
                  off->numel() == start.numel() &&
                  len->numel() == start.numel(), "per-portion arrays");
  st.item = item->data_ptr<int>(); st.t0 = t0->data_ptr<int>();
  st.off = off->data_ptr<int>(); st.len = len->data_ptr<int>();
  return (int)item->numel();
}

static void chk_conv(const Tensor& x, const Tensor& w, const Tensor& tails,
                     long C) {
  CHK_DEV(x); chk_rows(x, "x"); CHK_F32(w); CHK_CONT(tails);
  CHK_SAME(x, tails);
  TORCH_CHECK(w.dim() == 2 && w.size(1) == C, "filters [taps, C]");
  TORCH_CHECK(w.size(0) >= 1 && w.size(0) <= 17, "1 to 17 taps");
  TORCH_CHECK(tails.dim() == 3 && tails.size(1) == w.size(0) - 1 &&
                  tails.size(2) == C, "tails [slots, taps - 1, C]");
  TORCH_CHECK(x.size(1) >= C, "columns");
}

// x columns [q | k | v] to rotated q [T, H*D], k and v to their pages: what the
// kernels take, without the step
static ConvQkv conv_qkv_args(const Tensor& x, const Tensor& w,
                             const Tensor& tails, const Tensor& cos_t,
                             const Tensor& sin_t, long rot,
                             const Tensor& cache_slots, const Tensor& kc,
                             const Tensor& vc, long H, Tensor& q, int* v4) {
  CHK_CONT(kc); CHK_CONT(vc); CHK_SAME(x, kc); CHK_SAME(x, vc);
  CHK_I32(cache_slots);
  TORCH_CHECK(kc.dim() == 4 && kc.size(2) == 64 && vc.dim() == 4 &&
                  vc.size(2) == 64 && vc.size(0) == kc.size(0) &&
                  vc.size(1) == kc.size(1), "pages [P, G, 64, D], [P, G, 64, E]");
  const int G = (int)kc.size(1), D = (int)kc.size(3), E = (int)vc.size(3);
  const long C = (H + G) * (long)D + (long)G * E;
  chk_conv(x, w, tails, C);
  TORCH_CHECK(rot % 2 == 0 && rot >= 0 && rot <= D, "rotated dims");
  int table_len = 0x7fffffff;
  if (rot > 0) {
    CHK_F32(cos_t); CHK_F32(sin_t);
    TORCH_CHECK(cos_t.dim() == 2 && cos_t.size(1) == rot / 2 &&
                    sin_t.sizes() == cos_t.sizes() && cos_t.size(0) > 0,
                "rotation tables");
    table_len = (int)cos_t.size(0);
  }
  const long T = x.size(0);
  TORCH_CHECK(cache_slots.numel() == T, "one cache slot per row");
  q = torch::empty({T, H * (long)D}, x.options());
  *v4 = D % 4 == 0 && E % 4 == 0 && rot % 8 == 0 && x.stride(0) % 4 == 0 &&
        aligned(x, is_f32(x) ? 16 : 8);
  return ConvQkv{x.data_ptr(), x.stride(0), w.data_ptr<float>(),
                 (int)w.size(0), tails.data_ptr(), ConvStep{},
                 rot ? cos_t.data_ptr<float>() : nullptr,
                 rot ? sin_t.data_ptr<float>() : nullptr, (int)rot, table_len,
                 cache_slots.data_ptr<int>(), q.data_ptr(), kc.data_ptr(),
                 vc.data_ptr(), (int)H, G, D, E};
}

Tensor conv_qkv(Tensor x, Tensor w, Tensor tails, Tensor cos_t, Tensor sin_t,
                long rot, Tensor cache_slots, Tensor kc, Tensor vc, long H,
                OptTensor item, OptTensor t0, OptTensor off, Tensor start,
                OptTensor len, Tensor slots) {
  Tensor q;
  int v4;
  ConvQkv p = conv_qkv_args(x, w, tails, cos_t, sin_t, rot, cache_slots, kc,
                            vc, H, q, &v4);
  if (x.size(0) == 0) return q;
  const int chunks = conv_step(p.step, item, t0, off, start, len, slots,
                               x.size(0));
  qsa_conv_qkv_launch(p, x.size(0), chunks, is_f32(x), v4, cur_stream());
  return q;
}

// silu(conv(x) + bias) -> dense [T, C]
Tensor conv_silu(Tensor x, Tensor w, Tensor bias, Tensor tails,
                 OptTensor item, OptTensor t0, OptTensor off, Tensor start,
                 OptTensor len, Tensor slots) {
  const long T = x.size(0), C = x.size(1);
  chk_conv(x, w, tails, C);
  CHK_F32(bias);
  TORCH_CHECK(bias.numel() == C, "bias");
  auto out = torch::empty({T, C}, x.options());
  if (T == 0) return out;
  ConvStep st;
  const int chunks = conv_step(st, item, t0, off, start, len, slots, T);
  const int v4 = C % 4 == 0 && x.stride(0) % 4 == 0 &&
                 aligned(x, is_f32(x) ? 16 : 8);
  qsa_conv_silu_launch(x.data_ptr(), x.stride(0), w.data_ptr<float>(),
                       bias.data_ptr<float>(), (int)w.size(0),
                       tails.data_ptr(), st, x.size(0), chunks,
                       out.data_ptr(), (int)C, is_f32(x), v4, cur_stream());
  return out;
}

// ---- grouped-query attention over pages ------------------------------------
struct GqaDims { int R, H, G, D, E; };

static GqaDims gqa_check(const Tensor& q, const Tensor& kc, const Tensor& vc,
                         const Tensor& block_table, const OptTensor& sink,
                         const OptTensor& gate, const Tensor& out, long H) {
  CHK_DEV(q); CHK_CONT(q); CHK_CONT(kc); CHK_CONT(vc); CHK_SAME(q, kc);
  CHK_SAME(q, vc); CHK_SAME(q, out); chk_rows(out, "out");
  CHK_I32(block_table);
  TORCH_CHECK(block_table.dim() == 2, "block_table [items, pages]");
  TORCH_CHECK(kc.dim() == 4 && kc.size(2) == 64 && vc.dim() == 4 &&
                  vc.size(2) == 64 && vc.size(0) == kc.size(0) &&
                  vc.size(1) == kc.size(1), "pages [P, G, 64, D], [P, G, 64, E]");
  GqaDims d{(int)q.size(0), (int)H, (int)kc.size(1), (int)kc.size(3),
            (int)vc.size(3)};
  TORCH_CHECK(q.dim() == 2 && q.size(1) == H * d.D, "q [R, H*D]");
  TORCH_CHECK(d.G > 0 && H % d.G == 0, "query heads per key head");
  TORCH_CHECK(out.size(0) == d.R && out.size(1) == H * d.E, "out [R, H*E]");
  if (sink) {
    CHK_F32(*sink);
    TORCH_CHECK(sink->numel() == H, "one sink per head");
  }
  if (gate) {
    CHK_SAME(q, *gate); chk_rows(*gate, "gate");
    TORCH_CHECK(gate->size(0) == d.R && gate->size(1) == H * d.E, "gate");
  }
  return d;
}

bool gqa_mfma_ok(long D, long E) {
  return D <= 256 && E <= 256 && D % 8 == 0 && E % 8 == 0;
}

static bool gqa_aligned(const Tensor& q, const OptTensor& gate,
                        const Tensor& out) {
  return aligned(q, 16) && out.stride(0) % 4 == 0 && aligned(out, 8) &&
         (!gate || (gate->stride(0) % 4 == 0 && aligned(*gate, 8)));
}

// q [R, H*D] rows -> rows of out; row_item: which block_table row a query row
// uses (none: its own index); row_len: position + 1 (0: row not in use)
// A row may be finished by the block, as four shares, which saves the partial
// results and a launch: where rows fill the chip so, or are over before the merge
// would start; where they are so many or so short that a wave each is enough,
// three of its four waves are in the way.  us, shares and a merge kernel / in the
// block, 16 heads of 128 on 8:
//   1 row (8 tiles), 20-60 keys 9.1 / 5.7, 300-500 11.2 / 9.3, 500-1000 11.1 / 13.9
//   15 rows (120)               9.8 / 5.8,         13.7 / 10.2,         19.6 / 20.6
//   17 rows (136)              10.0 / 5.9,         16.6 / 11.0,         23.5 / 20.5
//   24 rows (192), 500-1000 27.6 / 21.6, 1000-2000 40.2 / 35.2, 3000-4096 77 / 69
//   17 rows (136)           23.5 / 20.5,           34.3 / 33.6,           58 / 62
// and of many:
//    64 rows (512 tiles), 10-60 keys 10.5 /  7.4, 400-1000 37.5 / 34.1
//   256 rows (2048)            14.0 / 20.9,                79.9 / 71.7
//   1024 rows (8192)           39.6 / 71.6,                 264 / 250
// 50-300 keys, a table of five pages: 192 rows 33.9 / 31.0, 512 50.5 / 60.4; of
// heads of 64: 512 rows 29.7 / 26.7, 1024 49.9 / 50.6.  Heads beyond 128 leave
// one block a CU: 17 heads on 1 of 256 / 136, 300 rows (600 tiles) of 50-300 34
// / 41, 512 rows of 400-1000 100 / 109; 16 on 4 of 192 / 128, 128 rows of
// 50-300 (512) 26.7 / 21.6, 192 of 400-1000 (768) 90 / 76, 512 (2048) 136 / 141.
// mp: the table's columns, as the rows' lengths are on the device.
static bool gqa_merge_in_block(long long tiles, int mp, int D, int E) {
  const int wide = std::max(D, E);
  if (tiles < 512)
    return wide <= 128 &&
           (mp <= 8 || tiles >= 192 || (mp <= 16 && tiles >= 129));
  if (wide > 128)
    return tiles == 512 || (mp >= 8 && tiles <= (E <= 128 ? 1600 : 800));
  if (tiles <= 1024 || mp >= 8) return true;
  return mp >= 4 && (wide <= 64 || tiles <= 2048);
}

void gqa_rows(Tensor q, Tensor kc, Tensor vc, Tensor block_table,
              OptTensor row_item, Tensor row_len, OptTensor sink,
              OptTensor gate, Tensor out, long H, double scale,
              double out_scale) {
  const GqaDims d = gqa_check(q, kc, vc, block_table, sink, gate, out, H);
  CHK_I32(row_len);
  TORCH_CHECK(row_len.numel() == d.R, "row arrays");
  const int* ri = nullptr;
  if (row_item) {
    CHK_I32(*row_item);
    TORCH_CHECK(row_item->numel() == d.R, "row_item");
    ri = row_item->data_ptr<int>();
  } else {
    TORCH_CHECK(block_table.size(0) >= d.R, "block_table rows");
  }
  if (d.R == 0) return;
  const int mp = (int)block_table.size(1);
  const int f32 = is_f32(q);
  const float* sp = sink ? sink->data_ptr<float>() : nullptr;
  const void* gp = gate ? gate->data_ptr() : nullptr;
  const long long gs = gate ? gate->stride(0) : 0;
  if (!f32 && gqa_mfma_ok(d.D, d.E) && gqa_aligned(q, gate, out)) {
    const long long tiles =
        (long long)d.R * d.G * ((d.H / d.G + 15) / 16);
    // two waves a SIMD fill the chip; no shares that differ by a page when
    // they need not
    const bool merge = gqa_merge_in_block(tiles, mp, d.D, d.E);
    long long ns = 4;
    if (!merge) {
      ns = (2048 + tiles - 1) / tiles;
      const long long pages = std::max(mp, 1);       // none: rows not in use
      ns = std::min(ns, pages);
      const long long per = (pages + ns - 1) / ns;
      ns = (pages + per - 1) / per;
    }
    TORCH_CHECK(tiles * ns < (1LL << 31), "rows per call");
    auto of = q.options().dtype(at::kFloat);
    Tensor po, pm;
    if (!merge) {
      po = torch::empty({d.R, d.H, ns, d.E}, of);
      pm = torch::empty({d.R, d.H, ns, 2}, of);
    }
    qsa_gqa_rows_mfma_launch(
        u16(q), u16(kc), u16(vc), block_table.data_ptr<int>(), mp, ri,
        row_len.data_ptr<int>(), sp, (const bf16_t*)gp, gs,
        merge ? nullptr : po.data_ptr<float>(),
        merge ? nullptr : pm.data_ptr<float>(), u16m(out), out.stride(0),
        d.R, d.H, d.G, d.D, d.E, (float)scale, (float)out_scale, (int)ns,
        cur_stream());
  } else {
    TORCH_CHECK(d.D + d.E <= 12000, "head too wide");
    qsa_gqa_rows_launch(q.data_ptr(), kc.data_ptr(), vc.data_ptr(),
                        block_table.data_ptr<int>(), mp, ri,
                        row_len.data_ptr<int>(), sp, gp, gs, out.data_ptr(),
                        out.stride(0), d.R, d.H, d.G, d.D, d.E, (float)scale,
                        (float)out_scale, f32, cur_stream());
  }
}

// query rows a block of gqa_portions takes
long gqa_portion_rows(long D, long E) {
  return D <= 128 && E <= 128 ? 128 : 64;
}

// portions' rows of q; block_table row i belongs to portion i
void gqa_portions(Tensor q, Tensor kc, Tensor vc, Tensor block_table,
                  OptTensor sink, OptTensor gate, Tensor qb_item,
                  Tensor qb_t0, Tensor off, Tensor start, Tensor len,
                  Tensor out, long H, double scale, double out_scale) {
  const GqaDims d = gqa_check(q, kc, vc, block_table, sink, gate, out, H);
  TORCH_CHECK(q.scalar_type() == at::kBFloat16, "bf16 storage");
  TORCH_CHECK(gqa_mfma_ok(d.D, d.E) && gqa_aligned(q, gate, out),
              "head sizes and alignment of the matrix-core path");
  CHK_I32(qb_item); CHK_I32(qb_t0); CHK_I32(off); CHK_I32(start);
  CHK_I32(len);
  const int QB = (int)qb_item.numel();
  const auto n = off.numel();
  TORCH_CHECK(qb_t0.numel() == QB && start.numel() == n && len.numel() == n &&
                  block_table.size(0) == n, "plan arrays");
  if (QB == 0) return;
  qsa_gqa_portions_launch(
      u16(q), u16(kc), u16(vc), block_table.data_ptr<int>(),
      (int)block_table.size(1), sink ? sink->data_ptr<float>() : nullptr,
      gate ? u16(*gate) : nullptr, gate ? gate->stride(0) : 0,
      qb_item.data_ptr<int>(), qb_t0.data_ptr<int>(), off.data_ptr<int>(),
      start.data_ptr<int>(), len.data_ptr<int>(), u16m(out), out.stride(0),
      QB, d.H, d.G, d.D, d.E, (float)scale, (float)out_scale,
      gqa_portion_rows(d.D, d.E) == 128, cur_stream());
}

// ---- state-space duality ---------------------------------------------------
struct SsdDims { int H, N, P, G; };

static SsdDims ssd_check(const Tensor& u, const Tensor& xbc, const Tensor& A,
                         const Tensor& dt_bias, const Tensor& D,
                         const Tensor& state, const Tensor& out, long G,
                         long zoff, long dtoff) {
  CHK_DEV(u); chk_rows(u, "u"); CHK_CONT(xbc); CHK_CONT(out);
  CHK_SAME(u, xbc); CHK_SAME(u, out); CHK_F32(A); CHK_F32(dt_bias);
  CHK_F32(D); CHK_F32(state);
  TORCH_CHECK(state.dim() == 4, "state [slots, H, N, P]");
  SsdDims s{(int)state.size(1), (int)state.size(2), (int)state.size(3),
            (int)G};
  const long inner = (long)s.H * s.P;
  TORCH_CHECK(G > 0 && s.H % G == 0, "heads per group");
  TORCH_CHECK(A.numel() == s.H && dt_bias.numel() == s.H &&
                  D.numel() == s.H, "per-head constants");
  TORCH_CHECK(xbc.dim() == 2 && xbc.size(0) == u.size(0) &&
                  xbc.size(1) == inner + 2 * G * s.N, "xbc [T, x | B | C]");
  TORCH_CHECK(out.dim() == 2 && out.size(0) == u.size(0) &&
                  out.size(1) == inner, "out [T, H*P]");
  TORCH_CHECK(zoff >= 0 && zoff + inner <= u.size(1) && dtoff >= 0 &&
                  dtoff + s.H <= u.size(1), "columns of z and dt");
  return s;
}

Tensor ssd_decode(Tensor u, long zoff, long dtoff, Tensor xbc, Tensor A,
                  Tensor dt_bias, Tensor D, Tensor state, long G,
                  Tensor slots, Tensor seq_lens) {
  auto out = torch::empty({u.size(0), state.size(1) * state.size(3)},
                          u.options());
  const SsdDims s = ssd_check(u, xbc, A, dt_bias, D, state, out, G, zoff,
                              dtoff);
  CHK_I32(slots); CHK_I32(seq_lens);
  const int B = (int)u.size(0);
  TORCH_CHECK(slots.numel() == B && seq_lens.numel() == B, "slots/seq_lens");
  TORCH_CHECK(s.N <= 5000, "state too wide for the decode block");
  if (B == 0) return out;
  const int a = is_f32(u) ? 16 : 8;
  const int v4 = s.P % 4 == 0 && xbc.size(1) % 4 == 0 && zoff % 4 == 0 &&
                 u.stride(0) % 4 == 0 && aligned(u, a) && aligned(xbc, a);
  qsa_ssd_decode_launch(
      u.data_ptr(), u.stride(0), (int)zoff, (int)dtoff, xbc.data_ptr(),
      A.data_ptr<float>(), dt_bias.data_ptr<float>(), D.data_ptr<float>(),
      state.data_ptr<float>(), slots.data_ptr<int>(),
      seq_lens.data_ptr<int>(), out.data_ptr(), B, s.H, s.N, s.P, s.G,
      is_f32(u), v4, cur_stream());
  return out;
}

bool ssd_step_ok(long H, long N, long P, long G, long parts, long taps) {
  return qsa_ssd_step_rows((int)H, (int)N, (int)P, (int)G, (int)parts,
                           (int)taps) > 0;
}

// Single tokens of a parallel layer: x | u are columns of its projection's rows.  The
// attention's convolutions (returns q, writes k and v to their pages), and the whole
// state-space branch, its normed read-out to rows of out.
Tensor ssd_step(Tensor x, Tensor qw, Tensor qtails, Tensor cos_t, Tensor sin_t,
                long rot, Tensor cache_slots, Tensor kc, Tensor vc, long H,
                Tensor u, Tensor w, Tensor bias, Tensor tails, Tensor A,
                Tensor dt_bias, Tensor D, Tensor state, long G, Tensor norm,
                double eps, Tensor out, Tensor slots, Tensor seq_lens) {
  Tensor q;
  int v4;
  ConvQkv conv = conv_qkv_args(x, qw, qtails, cos_t, sin_t, rot,
                                     cache_slots, kc, vc, H, q, &v4);
  CHK_F32(state); CHK_F32(bias); CHK_F32(A); CHK_F32(dt_bias); CHK_F32(D);
  CHK_F32(norm); CHK_SAME(u, x); CHK_SAME(u, out);
  CHK_DEV(u); chk_rows(u, "u"); chk_rows(out, "out");
  chk_there(u, x, qw, qtails, cache_slots, kc, vc, w, bias, tails, A, dt_bias, D,
            state, norm, out, slots, seq_lens);
  if (rot) chk_there(u, cos_t, sin_t);
  TORCH_CHECK(u.scalar_type() == at::kBFloat16, "bf16 storage");
  TORCH_CHECK(state.dim() == 4, "state [slots, H, N, P]");
  const int SH = (int)state.size(1), N = (int)state.size(2),
            P = (int)state.size(3), B = (int)u.size(0);
  const long inner = (long)SH * P, C = inner + 2 * G * N;
  const Tensor xbc = u.narrow(1, inner, C);
  chk_conv(xbc, w, tails, C);
  TORCH_CHECK(ssd_step_ok(SH, N, P, G, G, w.size(0)) && conv.taps <= 4,
              "sizes of the step");
  TORCH_CHECK(bias.numel() == C && A.numel() == SH && dt_bias.numel() == SH &&
                  D.numel() == SH && norm.numel() == inner, "constants");
  TORCH_CHECK(x.size(0) == B && out.size(0) == B && out.size(1) == inner &&
                  u.size(1) >= inner + C + SH, "rows and columns");
  conv_step(conv.step, c10::nullopt, c10::nullopt,
            c10::nullopt, seq_lens, c10::nullopt, slots, B);
  TORCH_CHECK(v4 && u.stride(0) % 4 == 0 && aligned(u, 8) &&
                  out.stride(0) % 4 == 0 && aligned(out, 8) &&
                  aligned(norm, 16) && aligned(state, 16), "alignment");
  if (B == 0) return q;
  qsa_ssd_step_launch(
      SsdStep{u16(u), u.stride(0), 0, (int)inner, (int)(inner + C),
              w.data_ptr<float>(), bias.data_ptr<float>(), (int)w.size(0),
              u16m(tails), A.data_ptr<float>(), dt_bias.data_ptr<float>(),
              D.data_ptr<float>(), norm.data_ptr<float>(),
              state.data_ptr<float>(), slots.data_ptr<int>(),
              seq_lens.data_ptr<int>(), u16m(out), out.stride(0), B, SH, N, P,
              (int)G, (float)eps, 0, conv},
      cur_stream());
  return q;
}

void ssd_seq(Tensor u, long zoff, long dtoff, Tensor xbc, Tensor A,
             Tensor dt_bias, Tensor D, Tensor state, long G, Tensor slots,
             Tensor off, Tensor start, Tensor len, Tensor out) {
  const SsdDims s = ssd_check(u, xbc, A, dt_bias, D, state, out, G, zoff,
                              dtoff);
  const int n = chk_items(slots, off, start, len);
  TORCH_CHECK(s.N <= 5000, "state too wide");
  if (n == 0) return;
  qsa_ssd_seq_launch(
      u.data_ptr(), u.stride(0), (int)zoff, (int)dtoff, xbc.data_ptr(),
      A.data_ptr<float>(), dt_bias.data_ptr<float>(), D.data_ptr<float>(),
      state.data_ptr<float>(), slots.data_ptr<int>(), off.data_ptr<int>(),
      start.data_ptr<int>(), len.data_ptr<int>(), out.data_ptr(), n, s.H,
      s.N, s.P, s.G, is_f32(u), cur_stream());
}

bool ssd_chunked_ok(long H, long N, long P, long G) {
  return N <= 256 && P <= 256 && N % 8 == 0 && P % 8 == 0 && H % G == 0;
}

// chunked prefill of the portions (chunks of 64 tokens)
void ssd_chunked(Tensor u, long zoff, long dtoff, Tensor xbc, Tensor A,
                 Tensor dt_bias, Tensor D, Tensor state, long G, Tensor slots,
                 Tensor off, Tensor start, Tensor len, Tensor chunk0,
                 Tensor chunk_item, Tensor chunk_t0, Tensor out) {
  const SsdDims s = ssd_check(u, xbc, A, dt_bias, D, state, out, G, zoff,
                              dtoff);
  const int n = chk_items(slots, off, start, len);
  CHK_I32(chunk0); CHK_I32(chunk_item); CHK_I32(chunk_t0);
  TORCH_CHECK(u.scalar_type() == at::kBFloat16, "bf16 storage");
  TORCH_CHECK(ssd_chunked_ok(s.H, s.N, s.P, G), "sizes of the chunked path");
  TORCH_CHECK(zoff % 4 == 0 && u.stride(0) % 4 == 0 && aligned(u, 8) &&
                  aligned(xbc, 16), "alignment");
  const long long nc = chunk_item.numel();
  TORCH_CHECK(chunk0.numel() == n && chunk_t0.numel() == nc, "plan arrays");
  if (n == 0 || nc == 0) return;
  const int DP = pad_dim(s.N), EP = (s.P + 15) / 16 * 16;
  auto steps = torch::empty({nc, s.H, 2, 64}, u.options().dtype(at::kFloat));
  auto prefix = torch::empty({nc, s.H, 2, EP, DP}, u.options());
  hipStream_t st = cur_stream();
  qsa_ssd_steps_launch(u16(u), u.stride(0), (int)dtoff, A.data_ptr<float>(),
                       dt_bias.data_ptr<float>(), off.data_ptr<int>(),
                       len.data_ptr<int>(), chunk_item.data_ptr<int>(),
                       chunk_t0.data_ptr<int>(), steps.data_ptr<float>(),
                       (int)nc, s.H, st);
  qsa_ssd_state_launch(u16(xbc), steps.data_ptr<float>(),
                       state.data_ptr<float>(), slots.data_ptr<int>(),
                       off.data_ptr<int>(), start.data_ptr<int>(),
                       len.data_ptr<int>(), chunk0.data_ptr<int>(),
                       prefix.data_ptr(), n, s.H, s.N, DP, s.P, EP, s.G, st);
  qsa_ssd_out_launch(u16(u), u.stride(0), (int)zoff, u16(xbc),
                     steps.data_ptr<float>(), D.data_ptr<float>(),
                     off.data_ptr<int>(), start.data_ptr<int>(),
                     len.data_ptr<int>(), chunk_item.data_ptr<int>(),
                     chunk_t0.data_ptr<int>(), prefix.data_ptr(), (int)nc,
                     u16m(out), s.H, s.N, DP, s.P, EP, s.G, st);
}

// rms norm of `parts` equal parts of a row, times w -> rows of out
void part_norm(Tensor x, Tensor w, Tensor out, long parts, double eps) {
  CHK_DEV(x); CHK_CONT(x); CHK_F32(w); CHK_SAME(x, out);
  chk_rows(out, "out");
  TORCH_CHECK(x.dim() == 2 && out.sizes() == x.sizes() &&
                  w.numel() == x.size(1), "x, w, out shapes");
  TORCH_CHECK(parts > 0 && x.size(1) % parts == 0, "equal parts");
  const int n = (int)(x.size(1) / parts);
  if (x.numel() == 0) return;
  const int a = is_f32(x) ? 16 : 8;
  const int v = n % 4 == 0 && out.stride(0) % 4 == 0 && aligned(x, a) &&
                aligned(out, a);
  qsa_part_norm_launch(x.data_ptr(), w.data_ptr<float>(), out.data_ptr(),
                       out.stride(0), x.size(0), (int)parts, n, (float)eps,
                       is_f32(x), v, cur_stream());
}

// weight-streaming decode product, W packed as [N/16, K/32, 16, 32]
Tensor skinny_gemm(Tensor a, Tensor wf, long N, long K, bool far) {
  CHK_DEV(a); chk_rows(a, "a"); CHK_CONT(wf); CHK_SAME(a, wf);
  TORCH_CHECK(a.scalar_type() == at::kBFloat16, "bf16");
  const int M = (int)a.size(0);
  TORCH_CHECK(M >= 1 && M <= 32 && a.size(1) == K, "M in [1, 32], K");
  TORCH_CHECK(K % 256 == 0 && N % 16 == 0 && wf.numel() == N * K, "W packing");
  TORCH_CHECK(a.stride(0) % 8 == 0 && aligned(a, 16), "a alignment");
  // the kernel reads by descriptors: 32-bit offsets of whole 16 bytes
  if (M * a.stride(0) >= 1ll << 30) a = a.clone(at::MemoryFormat::Contiguous);
  if (!aligned(wf, 16)) wf = wf.clone(at::MemoryFormat::Contiguous);
  auto out = torch::empty({M, (long long)N}, a.options());
  qsa_skinny_gemm_launch(u16(a), u16(wf), u16m(out), M, (int)N, K,
                         a.stride(0), far, cur_stream());
  return out;
}

// Whether only the values of a tensor matter: derivatives in either direction,
// function transforms, traces, modes and autocast see the library's operations
// and would pass a kernel of our own by.
static bool unobserved(const Tensor& t) {
  using K = c10::DispatchKey;
  return !(at::GradMode::is_enabled() && t.requires_grad()) &&
         !t._fw_grad(0).defined() &&
         !t.key_set().has_any(c10::DispatchKeySet(
             {K::Python, K::FuncTorchBatched, K::FuncTorchGradWrapper,
              K::Batched, K::Functionalize, K::Conjugate, K::Negative,
              K::ZeroTensor}));
}

static bool no_observer() {
  return !c10::impl::tls_local_dispatch_key_set().included_.has(
             c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !at::tracer::impl::is_dispatch_enabled() &&
         !at::autocast::is_autocast_enabled(at::kCUDA);
}

// What rows_gemm.hip takes: bf16 with whole stages of K and column tiles, aligned
// rows, and offsets within a block's rows (and from a gate's weights to its
// up's) that fit 32 bits.
static bool rows_gemm_fits(const Tensor& a, const Tensor& w, bool glu) {
  if (a.dim() != 2 || w.dim() != 2) return false;
  const int64_t M = a.size(0), N = w.size(0), K = w.size(1), ld = a.stride(0);
  return M >= 1 && N >= 16 && K >= 64 && N % (glu ? 32 : 16) == 0 &&
         K % 64 == 0 && a.size(1) == K && M < 1 << 24 && N < 1 << 24 &&
         K < 1 << 24 && a.scalar_type() == at::kBFloat16 &&
         w.scalar_type() == at::kBFloat16 && w.is_contiguous() &&
         a.stride(1) == 1 && ld % 8 == 0 && ld >= 0 && ld < 1 << 24 &&
         (std::min<int64_t>(M, 256) * ld + K) * 2 < (4ll << 30) &&
         ((glu ? N / 2 : 0) + 257) * K * 2 < (4ll << 30) && aligned(a, 16) &&
         aligned(w, 16);
}

// Whether a @ w^T, with `glu` the gated activation of it, is rows_gemm's by its
// sizes, before wide_gemm is looked at.  As plain products of 26 pairs of N and K with M
// of 33 to 14000 it is 18 % faster than the library's on average while M N is at most
// 9 million, and as 15 pairs with M of 1 to 32 13 % (6144 x 4096 alone, which the packed
// stream has, is up to 8 % behind).  With K up to 768 the library's are not yet in
// their stride: 8800 x 4096 x 512 takes 46 us for 75.  Beyond these lines, and gated
// beyond 48 million of longer K, wide_gemm is asked (wide_sizes) and, where it cannot,
// with fewer than 256 rows or rows too far apart, the library.
// The activation inside leaves K whole: where a plain product is this kernel's too and
// few blocks would split it, that and a launch for the activation
// is sooner (33 x 2048 x 16384 22 us, inside 69, the library 27; 64 x 4096 x 8192
// 21, 41, 27; 100 x 4096 x 2048 11.8, 10.9, 12.2).  Of 881 gated shapes that left
// 4 slower than inside, by up to 10 %, and takes 0.84 of the library's time on
// average, 0.93 with all inside.
static bool rows_gemm_sizes(int64_t M, int64_t N, int64_t K, bool glu) {
  const int64_t MN = M * N;
  const bool plain = MN <= 9000000 || K <= 768;
  if (!glu) return plain;
  if (MN > 48000000 && K > 3072) return false;
  if (!plain || K < 512) return true;  // beside the library's; not split
  int S;
  float in, apart;
  qsa_rows_gemm_plan((int)M, (int)N, (int)K, 1, 0, &S, &in);
  qsa_rows_gemm_plan((int)M, (int)N, (int)K, 0, 0, &S, &apart);
  return in <= apart + 4.f + 6.4e-7f * (float)MN;
}

// Such a call as a whole; one that is not captured is spared 15 us of the library's
// host path.  All of it is here: in Python the last part alone took 2 us a call.
static bool gemm_takes(const Tensor& a, const Tensor& w, bool glu) {
  return a.is_cuda() && a.device() == w.device() && no_observer() &&
         unobserved(a) && unobserved(w) && rows_gemm_fits(a, w, glu);
}

bool rows_gemm_ok(const Tensor& a, const Tensor& w) {
  return gemm_takes(a, w, false) &&
         rows_gemm_sizes(a.size(0), w.size(0), w.size(1), false);
}

bool rows_glu_ok(const Tensor& a, const Tensor& w) {
  return gemm_takes(a, w, true) &&
         rows_gemm_sizes(a.size(0), w.size(0), w.size(1), true);
}

// Whether wide_gemm.hip can do a product, whose first tile takes the shortest K; its
// offsets are of whole tiles.  Decode batches, bound by the read of W, are not looked
// at.
static bool wide_takes(int64_t M, int64_t N, int64_t K, int64_t lda, int act) {
  return M >= 256 && (256 * lda + K) * 2 < (4ll << 30) &&
         256 * N * 2 < (4ll << 30) && qsa_wide_gemm_fits(0, (int)K, act);
}

// Whether a product is wide_gemm.hip's where it is not rows_gemm.hip's by its size.
// With the activation, a pass of its own beside the library's product, it takes 0.91
// of that time (157 products of M 300 to 30,000), at most 1.02.  Plain ones take 0.93
// (260 of M 256 to 46,000), but which way depends on the library, that is uneven:
// 0.50 (3000 x 3584 x 18944) to 1.13.  It is ahead where tiles of 256 x 256 come in whole
// turns of the 256 CUs: there 77 products took 1.04 of its time (8192 x 4096 x 4096
// 178 / 186 us, 20,480 x 8192 x 8192 1753 / 1849; of K up to 1024 0.99), and these stay
// with it.  Left are 1.05 to 1.13 in 30 of 260, full but for part of one turn (2048 x
// 28672 x 4096 328 / 363, 13,800 x 2048 x 8192 318 / 340), beside products as full that
// the library takes 1.1 to 1.7 times as long for (10,816 x 4096 x 4096, 7500 x 4096 x
// 14336, 20,000 x 4096 x 4096).
static bool wide_sizes(int64_t M, int64_t N, int64_t K, int64_t lda, bool glu) {
  const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256);
  return M * N > 9000000 && (glu || K <= 1024 || tiles % 256) &&
         wide_takes(M, N, K, lda, glu);
}

// Whether a product of these sizes is one of the two's.
static bool gemm_sizes(int64_t M, int64_t N, int64_t K, int64_t lda, bool glu) {
  return rows_gemm_sizes(M, N, K, glu) || wide_sizes(M, N, K, lda, glu);
}

bool gemm_ok(const Tensor& a, const Tensor& w) {
  return gemm_takes(a, w, false) &&
         gemm_sizes(a.size(0), w.size(0), w.size(1), a.stride(0), false);
}

bool glu_gemm_ok(const Tensor& a, const Tensor& w) {
  return gemm_takes(a, w, true) &&
         gemm_sizes(a.size(0), w.size(0), w.size(1), a.stride(0), true);
}

// How a product is run.  wide: wide_gemm's tile, the rows that it takes and the tile of
// the rest; else rows_gemm's tile and shares of K.
struct GemmPlan {
  bool wide = false;
  int tile = 0, rows = 0, rest = 0, shares = 1;
};

// Whichever of the two should be over first, each asked once.  rows_gemm's estimate is
// of CUs that keep their clock: where it comes within 14 % of the other's, the other is
// sooner (of 200 shapes, M 200 to 45,000, the choice is then 0.5 % from the best).
static GemmPlan gemm_choice(int64_t M, int64_t N, int64_t K, int64_t lda, int act,
                            bool parts) {
  GemmPlan p;
  float rows_us, wide_us = 1e30f;
  p.tile = qsa_rows_gemm_plan((int)M, (int)N, (int)K, act, parts, &p.shares, &rows_us);
  if (!wide_takes(M, N, K, lda, act)) return p;
  int tile;
  wide_us = qsa_wide_gemm_plan((int)M, (int)N, (int)K, act, &tile, &p.rows, &p.rest);
  p.wide = wide_us < 1e30f && rows_us * 1.14f >= wide_us;
  if (p.wide) p.tile = tile;
  return p;
}

static void chk_product(const Tensor& a, const Tensor& w, int act) {
  CHK_DEV(a); CHK_SAME(a, w);
  TORCH_CHECK(rows_gemm_fits(a, w, act != 0), "bf16 a [M, K], w [N, K] with K % "
              "64 and N % 16 (gated: 32), aligned rows less than 2^24 apart");
}

// parts: a product whose K is split may stay in its shares, [S, M, N] f32; far: w is
// read past the last-level cache, where each of its numbers is read once
static Tensor rows_gemm_by(const Tensor& a, const Tensor& w, int act, bool parts,
                           bool far, int tile, int S) {
  const int M = (int)a.size(0), N = (int)w.size(0), K = (int)w.size(1);
  Tensor out, part;
  if (S > 1) part = torch::empty({S, M, N}, a.options().dtype(at::kFloat));
  if (S == 1 || !parts) out = torch::empty({M, act ? N / 2 : N}, a.options());
  qsa_rows_gemm_launch(u16(a), u16(w), out.defined() ? u16m(out) : nullptr,
                       S > 1 ? part.data_ptr<float>() : nullptr, M, N, K,
                       a.stride(0), tile, S, act, far, cur_stream());
  return out.defined() ? out : part;
}

static Tensor rows_gemm_run(const Tensor& a, const Tensor& w, int act,
                            bool parts = false, bool far = false) {
  chk_product(a, w, act);
  int S;
  const int tile = qsa_rows_gemm_plan((int)a.size(0), (int)w.size(0),
                                      (int)w.size(1), act, parts, &S, nullptr);
  return rows_gemm_by(a, w, act, parts, far, tile, S);
}

static Tensor gemm_run(const Tensor& a, const Tensor& w, int act, bool parts,
                       bool far) {
  chk_product(a, w, act);
  const int M = (int)a.size(0), N = (int)w.size(0), K = (int)w.size(1);
  const GemmPlan p = gemm_choice(M, N, K, a.stride(0), act, parts);
  if (!p.wide) return rows_gemm_by(a, w, act, parts, far, p.tile, p.shares);
  const int64_t cols = act ? N / 2 : N;
  Tensor out = torch::empty({M, cols}, a.options());
  qsa_wide_gemm_launch(u16(a), u16(w), u16m(out), p.rows, N, K, a.stride(0), p.tile,
                       act, cur_stream());
  if (p.rows < M)
    qsa_wide_gemm_launch(u16(a) + p.rows * a.stride(0), u16(w),
                         u16m(out) + p.rows * cols, M - p.rows, N, K, a.stride(0),
                         p.rest, act, cur_stream());
  return out;
}

// (tile, its rows, the tile of the rest) that the rule in wide_gemm.hip takes
std::tuple<int, int, int> wide_gemm_plan(int64_t M, int64_t N, int64_t K,
                                         bool glu) {
  int tile = -1, rows, rest;
  if (qsa_wide_gemm_plan((int)M, (int)N, (int)K, glu, &tile, &rows, &rest) == 1e30f)
    tile = -1;
  return {tile, rows, rest};
}

// the same of a product as gemm() and glu_gemm() run it; -1: rows_gemm's
std::tuple<int, int, int> gemm_plan(int64_t M, int64_t N, int64_t K, bool glu) {
  const GemmPlan p = gemm_choice(M, N, K, K, glu, false);
  return {p.wide ? p.tile : -1, p.rows, p.rest};
}

// a @ w^T by a tile of wide_gemm.hip, with act as in glu_gemm's kernels
Tensor wide_gemm(Tensor a, Tensor w, int64_t tile, int64_t act) {
  CHK_DEV(a); CHK_SAME(a, w);
  TORCH_CHECK(rows_gemm_fits(a, w, act != 0) && act >= 0 && act <= 3,
              "bf16 a [M, K], w [N, K] with K % 64 and N % 16 (gated: 32)");
  const int M = (int)a.size(0), N = (int)w.size(0), K = (int)w.size(1);
  TORCH_CHECK(qsa_wide_gemm_fits((int)tile, K, (int)act) &&
                  (256 * a.stride(0) + K) * 2 < (4ll << 30) &&
                  256ll * N * 2 < (4ll << 30), "tile, K and strides");
  Tensor out = torch::empty({M, act ? N / 2 : N}, a.options());
  qsa_wide_gemm_launch(u16(a), u16(w), u16m(out), M, N, K, a.stride(0), (int)tile,
                       (int)act, cur_stream());
  return out;
}

// (tile, shares of K) that the rule in rows_gemm.hip takes
std::tuple<int, int> rows_gemm_plan(int64_t M, int64_t N, int64_t K,
                                    bool glu) {
  int S;
  const int tile = qsa_rows_gemm_plan((int)M, (int)N, (int)K, glu, 0, &S,
                                      nullptr);
  return {tile, S};
}

// a @ w^T on W as it is stored.  These run rows_gemm.hip whatever the size, for its
// tests and for comparisons; models go through gemm() and its like below.
Tensor rows_gemm(Tensor a, Tensor w, bool far) {
  return rows_gemm_run(a, w, 0, false, far);
}

// the same for a reader that adds shares: [M, N], or [S, M, N] in f32
Tensor rows_parts(Tensor a, Tensor w) { return rows_gemm_run(a, w, 0, true); }

// res [rows, W] bf16 <- res + the sum of shares [S, rows, W], in place; returns
// rms norm of it times w
Tensor rmsnorm_shares(Tensor parts, Tensor res, Tensor w, double eps) {
  CHK_DEV(res); CHK_CONT(res); CHK_CONT(w); CHK_SAME(res, w);
  const int64_t W = res.size(-1), rows = W ? res.numel() / W : 0;
  TORCH_CHECK(is_shares(parts, res, rows, W) && w.numel() == W && W <= 8192 &&
                  aligned(res, 16) && aligned(w, 16), "shares, W <= 8192");
  auto out = torch::empty_like(res);
  if (rows)
    qsa_rmsnorm_shares_launch(parts.data_ptr<float>(), (int)parts.size(0),
                              u16m(res), u16(w), u16m(out), rows, (int)W,
                              (float)eps, cur_stream());
  return out;
}

// act of the first half of a @ w^T's columns times the second, of the products
// as they would be stored or (silu) of their sums
Tensor rows_glu(Tensor a, Tensor w, bool gelu, bool rounded) {
  TORCH_CHECK(rounded || !gelu, "gelu of the stored products only");
  return rows_gemm_run(a, w, gelu ? 2 : rounded ? 1 : 3);
}

// a @ w^T, for a reader that adds shares perhaps in them, and the gated activation of
// it, by whichever kernel the rules give
Tensor gemm(Tensor a, Tensor w, bool far) {
  return gemm_run(a, w, 0, false, far);
}
Tensor gemm_parts(Tensor a, Tensor w, bool far) {
  return gemm_run(a, w, 0, true, far);
}
Tensor glu_gemm(Tensor a, Tensor w, bool gelu, bool rounded, bool far) {
  TORCH_CHECK(rounded || !gelu, "gelu of the stored products only");
  return gemm_run(a, w, gelu ? 2 : rounded ? 1 : 3, false, far);
}

// ---- encoder ----------------------------------------------------------------

// A product of the encoder, planned once for all layers: short_gemm.hip's, or as gemm()
// and its like run it.
struct EncoderProduct {
  bool brief = false;
  GemmPlan plan;
  int M, N, K, act;

  bool set(const Tensor& a, const Tensor& w, bool glu, bool parts) {
    if (!gemm_takes(a, w, glu)) return false;
    const int64_t m = a.size(0), n = w.size(0), k = w.size(1);
    M = (int)m, N = (int)n, K = (int)k, act = glu ? 3 : 0;
    brief = qsa_short_gemm_takes(m, n, k);
    if (brief) return true;
    if (!gemm_sizes(m, n, k, a.stride(0), glu)) return false;
    plan = gemm_choice(m, n, k, a.stride(0), act, parts);
    return true;
  }
  int shares() const { return brief || plan.wide ? 1 : plan.shares; }
  int64_t part_size() const { return shares() > 1 ? (int64_t)shares() * M * N : 0; }
  void run(const Tensor& a, const Tensor& w, bf16_t* out, float* part,
           hipStream_t st) const {
    const long long lda = a.stride(0);
    if (brief) {
      qsa_short_gemm_launch(u16(a), u16(w), out, M, N, K, lda, act != 0, st);
    } else if (!plan.wide) {
      qsa_rows_gemm_launch(u16(a), u16(w), out, shares() > 1 ? part : nullptr, M, N, K,
                           lda, plan.tile, plan.shares, act, false, st);
    } else {
      const int64_t cols = act ? N / 2 : N;
      qsa_wide_gemm_launch(u16(a), u16(w), out, plan.rows, N, K, lda, plan.tile, act,
                           st);
      if (plan.rows < M)
        qsa_wide_gemm_launch(u16(a) + plan.rows * lda, u16(w), out + plan.rows * cols,
                             M - plan.rows, N, K, lda, plan.rest, act, st);
    }
  }
};

// The layers of the retrieval encoder on rows res [T, H], which they change, and the
// norm behind them; weights: attention's norm and feed-forward's, q k v, output,
// [gate; up] and down of every layer.  The kernels and their choice are those of the
// calls one by one (models/encoder.py), which are for all that this does not take: then
// there is no result and nothing has changed.  Up to some 2000 rows a call is as long as
// the host takes for its launches: 84 calls from Python at 5 us each, products planned
// each time; here they are planned once, and operands lie in the same places in every
// layer (texts embedded in one call, us: one of 15 tokens 520 -> 393, 8 of some 50 574 ->
// 503, from some 1000 tokens on level).  The price is that nothing takes another's place
// meanwhile: beside res 2 H + 4 A + F numbers of 16 bits a row, and the largest shares,
// 9 KB a row for the widths of EncoderConfig.
OptTensor encoder_layers(Tensor res, std::vector<Tensor> weights, Tensor final_norm,
                         Tensor cos_t, Tensor sin_t, Tensor qb_item, Tensor qb_t0,
                         Tensor off, Tensor len, int64_t heads, double scale,
                         double eps) {
  const size_t layers = weights.size() / 6;
  if (layers == 0 || weights.size() % 6 || !res.is_cuda() || res.dim() != 2 ||
      res.scalar_type() != at::kBFloat16 || !res.is_contiguous() || res.size(0) == 0 ||
      !aligned(res, 16) || !no_observer() || !unobserved(res) || heads <= 0 ||
      heads % 4)
    return c10::nullopt;
  const int64_t T = res.size(0), H = res.size(1), A = weights[3].size(-1),
                F = weights[5].size(-1), D = A / heads;
  if (H % 8 || H > 8192 || A % heads || (D != 64 && D != 128)) return c10::nullopt;
  auto norm_ok = [&](const Tensor& w) {
    return w.dim() == 1 && w.size(0) == H && w.is_contiguous() && aligned(w, 16) &&
           w.scalar_type() == at::kBFloat16 && w.device() == res.device() &&
           unobserved(w);
  };
  auto weight_ok = [&](const Tensor& w, int64_t n, int64_t k) {
    return w.dim() == 2 && w.size(0) == n && w.size(1) == k && w.is_contiguous() &&
           aligned(w, 16) && w.scalar_type() == at::kBFloat16 &&
           w.device() == res.device() && unobserved(w);
  };
  auto layer_ok = [&](size_t i) {
    const Tensor* w = &weights[i * 6];
    return norm_ok(w[0]) && norm_ok(w[1]) && weight_ok(w[2], 3 * A, H) &&
           weight_ok(w[3], H, A) && weight_ok(w[4], 2 * F, H) && weight_ok(w[5], H, F);
  };
  if (!norm_ok(final_norm) || !layer_ok(0)) return c10::nullopt;
  CHK_F32(cos_t); CHK_F32(sin_t);
  CHK_I32(qb_item); CHK_I32(qb_t0); CHK_I32(off); CHK_I32(len);
  chk_there(res, cos_t, sin_t, qb_item, qb_t0, off, len);
  TORCH_CHECK(cos_t.dim() == 2 && cos_t.size(0) >= 1 && cos_t.size(1) == D / 2 &&
                  sin_t.sizes() == cos_t.sizes(), "cos/sin [positions, D/2]");
  TORCH_CHECK(qb_item.numel() == qb_t0.numel() && off.numel() == len.numel(), "maps");
  const hipStream_t st = cur_stream();
  Tensor h = torch::empty_like(res);
  qsa_rmsnorm_launch(u16(res), u16(weights[0]), u16m(h), nullptr, T, (int)H, (float)eps,
                     st);
  // Until a product has been added to res nothing has changed: what the first layer
  // does before that is under way while the rest is looked at and planned.
  Tensor y = torch::empty_like(res);
  Tensor attn = torch::empty({T, A}, res.options());
  Tensor act = torch::empty({T, F}, res.options());
  Tensor qkv = torch::empty({T, 3 * A}, res.options());
  EncoderProduct p[4];
  Tensor part;
  auto space = [&](int q) {            // for the shares of product q
    if (p[q].part_size() > (part.defined() ? part.numel() : 0))
      part = torch::empty({p[q].part_size()}, res.options().dtype(at::kFloat));
  };
  auto shares = [&] { return part.defined() ? part.data_ptr<float>() : nullptr; };
  auto attention = [&](const Tensor* w) {
    p[0].run(h, w[2], u16m(qkv), shares(), st);
    qsa_encoder_attn_launch(u16(qkv), cos_t.data_ptr<float>(), sin_t.data_ptr<float>(),
                            (int)cos_t.size(0), qb_item.data_ptr<int>(),
                            qb_t0.data_ptr<int>(), off.data_ptr<int>(),
                            len.data_ptr<int>(), u16m(attn), (int)qb_item.numel(),
                            (int)heads, (int)D, (float)scale, st);
  };
  // a product for the norm behind it, which adds it to res and leaves the norm in h
  auto added = [&](int q, const Tensor& a, const Tensor& w, const Tensor& norm) {
    const bool split = p[q].shares() > 1;
    p[q].run(a, w, split ? nullptr : u16m(y), shares(), st);
    if (split)
      qsa_rmsnorm_shares_launch(shares(), p[q].shares(), u16m(res), u16(norm), u16m(h),
                                T, (int)H, (float)eps, st);
    else
      qsa_rmsnorm_launch(u16(y), u16(norm), u16m(h), u16m(res), T, (int)H, (float)eps,
                         st);
  };
  if (!p[0].set(h, weights[2], false, false)) return c10::nullopt;
  space(0);
  attention(&weights[0]);
  if (!p[1].set(attn, weights[3], false, true) || !p[2].set(h, weights[4], true, false) ||
      !p[3].set(act, weights[5], false, true))
    return c10::nullopt;
  for (size_t i = 1; i < layers; ++i)
    if (!layer_ok(i)) return c10::nullopt;
  for (int q = 1; q < 4; ++q) space(q);
  for (size_t i = 0; i < layers; ++i) {
    const Tensor* w = &weights[i * 6];
    if (i) attention(w);
    added(1, attn, w[3], w[1]);
    p[2].run(h, w[4], u16m(act), shares(), st);
    added(3, act, w[5], i + 1 < layers ? w[6] : final_norm);
  }
  return h;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("residual_norm", &residual_norm,
        "f32 residual update (+ embedding row, + vector) and layer/rms norm");
  m.def("glu", &glu, "act(gate) * up, bf16 or f32, any size");
  m.def("glu_table", &glu_table, "act(gate) * slice of the token's table row");
  m.def("conv_qkv", &conv_qkv,
        "short convolutions of q, k, v; rotation; k, v to their pages");
  m.def("conv_silu", &conv_silu, "short convolution with bias and silu");
  m.def("gqa_rows", &gqa_rows, "paged grouped-query attention of rows");
  m.def("gqa_portions", &gqa_portions,
        "paged grouped-query flash attention with sink and gate (MFMA)");
  m.def("gqa_mfma_ok", &gqa_mfma_ok, "size support");
  m.def("gqa_portion_rows", &gqa_portion_rows, "query rows per block");
  m.def("ssd_decode", &ssd_decode, "one token per row");
  m.def("ssd_step", &ssd_step,
        "single tokens of a parallel layer: convolutions, state and norm");
  m.def("ssd_step_ok", &ssd_step_ok, "size support");
  m.def("ssd_seq", &ssd_seq, "token loop over portions");
  m.def("ssd_chunked", &ssd_chunked, "chunked prefill (MFMA)");
  m.def("ssd_chunked_ok", &ssd_chunked_ok, "size support");
  m.def("part_norm", &part_norm, "rms norm in equal parts of a row");
  m.def("latent_norm_store", &latent_norm_store,
        "rms norms of the query and kv latents; kv latent to the cache");
  m.def("decode_slots", &decode_slots, "cache slot of each row's new position");
  m.def("argmax_rows", &argmax_rows, "greedy pick per row");
  m.def("retention_decode", &retention_decode, "one token per row");
  m.def("retention_seq", &retention_seq, "token loop over portions");
  m.def("retention_chunked", &retention_chunked, "chunked prefill (MFMA)");
  m.def("retention_chunked_ok", &retention_chunked_ok, "size support");
  m.def("head_matmul", &head_matmul, "per-head product (+ sigmoid gate)");
  m.def("latent_rows", &latent_rows, "absorbed latent attention of rows");
  m.def("window_attn_prefill", &window_attn_prefill,
        "windowed flash attention with sink and gate (MFMA)");
  m.def("window_attn_ok", &window_attn_ok, "size support");
  m.def("skinny_gemm", &skinny_gemm, "packed-weight decode GEMM (M <= 32)",
        py::arg("a"), py::arg("wf"), py::arg("N"), py::arg("K"),
        py::arg("far") = false);
  m.def("rows_gemm", &rows_gemm, "GEMM of decode batches and short prompts",
        py::arg("a"), py::arg("w"), py::arg("far") = false);
  m.def("rows_gemm_ok", &rows_gemm_ok, "whether a product is rows_gemm's");
  m.def("rows_parts", &rows_parts, "the same, shares of K left to the reader");
  m.def("rmsnorm_shares", &rmsnorm_shares,
        "residual add of such shares + RMSNorm (bf16)");
  m.def("rows_gemm_sizes", &rows_gemm_sizes,
        "whether sizes are rows_gemm's, or with the activation inside");
  m.def("rows_gemm_plan", &rows_gemm_plan, "tile and shares of a product");
  m.def("rows_glu", &rows_glu, "the same with the gated activation inside");
  m.def("rows_glu_ok", &rows_glu_ok, "whether a gated product is rows_glu's");
  m.def("gemm", &gemm, "rows_gemm or wide_gemm by size", py::arg("a"), py::arg("w"),
        py::arg("far") = false);
  m.def("gemm_ok", &gemm_ok, "whether a product is one of theirs");
  m.def("gemm_sizes", &gemm_sizes, "the same by its sizes and the rows' distance",
        py::arg("M"), py::arg("N"), py::arg("K"), py::arg("lda"), py::arg("glu"));
  m.def("gemm_parts", &gemm_parts, "the same, shares of K left to the reader",
        py::arg("a"), py::arg("w"), py::arg("far") = false);
  m.def("glu_gemm", &glu_gemm, "the same with the gated activation inside",
        py::arg("a"), py::arg("w"), py::arg("gelu"), py::arg("rounded"),
        py::arg("far") = false);
  m.def("glu_gemm_ok", &glu_gemm_ok, "whether a gated product is one of theirs");
  m.def("encoder_layers", &encoder_layers,
        "the layers of the retrieval encoder, or None: call by call");
  m.def("gemm_plan", &gemm_plan, "the same where gemm() takes wide_gemm, else -1");
  m.def("wide_gemm", &wide_gemm, "GEMM of many rows by a given tile");
  m.def("wide_gemm_plan", &wide_gemm_plan, "tiles and rows of a product");
}
