// Torch bindings for the qsa MI355X (gfx950) kernels.  HIP-native: no CUDA
// naming, no compatibility shims — this extension only builds for ROCm.
// Operator inventory these kernels implement: SURVEY.md 2.4 K1-K10
// (embedding, cosine top-k, anomaly scoring, paged-attention LLM decode,
// window aggregation, Avro wire codec).
#include <hip/hip_runtime.h>
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <pybind11/numpy.h>

#include <algorithm>
#include <cmath>

#define CHK(x) TORCH_CHECK(x, #x)
#define CHK_DEV(t) TORCH_CHECK((t).is_cuda(), #t " must be on the GPU")
#define CHK_CONT(t) TORCH_CHECK((t).is_contiguous(), #t " must be contiguous")
#define CHK_BF16(t) TORCH_CHECK((t).scalar_type() == at::kBFloat16, #t " must be bf16")
#define CHK_F32(t) TORCH_CHECK((t).scalar_type() == at::kFloat, #t " must be f32")
#define CHK_I32(t) TORCH_CHECK((t).scalar_type() == at::kInt, #t " must be i32")

static inline const unsigned short* u16(const torch::Tensor& t) {
  return reinterpret_cast<const unsigned short*>(t.data_ptr());
}
static inline unsigned short* u16m(torch::Tensor& t) {
  return reinterpret_cast<unsigned short*>(t.data_ptr());
}
static inline hipStream_t cur_stream() {
  return at::hip::getCurrentHIPStream().stream();
}

// ---- launcher decls (defined in the .hip files) ---------------------------
extern "C" void qsa_rmsnorm_launch(const unsigned short*, const unsigned short*,
                                   unsigned short*, unsigned short*, long long,
                                   int, float, hipStream_t);
extern "C" void qsa_swiglu_launch(const unsigned short*, const unsigned short*,
                                  unsigned short*, long long, long long,
                                  long long, int, hipStream_t);
extern "C" void qsa_rope_launch(unsigned short*, unsigned short*, const float*,
                                const float*, const int*, int, int, int, int,
                                long long, long long, hipStream_t);
extern "C" void qsa_softmax_rows_launch(float*, int, int, int, int, int,
                                        const int*, hipStream_t);
extern "C" void qsa_softmax_rows_bf16_launch(unsigned short*, long long, int,
                                             float, const int*, hipStream_t);
extern "C" void qsa_paged_attn_split(int, int, int, int, int, int*, int*);
extern "C" void qsa_paged_attn_mfma_launch(
    const unsigned short*, const unsigned short*, const unsigned short*,
    unsigned short*, unsigned short*, const float*, const float*, const int*,
    const int*, float*, float*, unsigned short*, float, int, int, int, int,
    int, long long, long long, int, int, int, const void* const*,
    const long long*, hipStream_t);
extern "C" void qsa_kv_append_launch(const unsigned short*,
                                     const unsigned short*, unsigned short*,
                                     unsigned short*, const int*, const int*,
                                     int, int, int, int, long long,
                                     hipStream_t);
extern "C" void qsa_paged_attn_prefill_launch(
    const unsigned short*, const unsigned short*, const unsigned short*,
    const int*, const int*, const int*, const int*, const int*, const int*,
    unsigned short*, float, int, int, int, int, int, long long, int, int,
    const float*, const float*, int,
    hipStream_t);
extern "C" void qsa_rope_kv_scatter_launch(
    unsigned short*, const unsigned short*, const unsigned short*,
    unsigned short*, unsigned short*, const float*, const float*, const int*,
    const int*, int, int, int, int, long long, long long, hipStream_t);
extern "C" void qsa_mean_rows_launch(const unsigned short*, const int*,
                                     const int*, float*, int, int,
                                     hipStream_t);
extern "C" void qsa_rope_kv_append_launch(unsigned short*,
                                          const unsigned short*,
                                          const unsigned short*,
                                          unsigned short*, unsigned short*,
                                          const float*, const float*,
                                          const int*, const int*, int, int,
                                          int, int, int, long long, long long,
                                          hipStream_t);
extern "C" void qsa_kv_scatter_launch(const unsigned short*,
                                      const unsigned short*, unsigned short*,
                                      unsigned short*, const int*, int, int,
                                      int, long long, hipStream_t);
extern "C" void qsa_skinny_gemm_launch(const unsigned short*,
                                       const unsigned short*, unsigned short*,
                                       int, int, long long, long long, bool,
                                       hipStream_t);
extern "C" int qsa_skinny_gemm_probe_launch(const unsigned short*,
                                            const unsigned short*,
                                            unsigned short*, int, int,
                                            long long, long long, int, int,
                                            hipStream_t);
extern "C" void qsa_skinny_gemm_fp8_launch(
    const unsigned short*, const unsigned char*, const float*,
    unsigned short*, unsigned short*, int, int, long long, long long, int,
    const unsigned short*, const float*, int, float, int, float*, int,
    hipStream_t);
extern "C" int qsa_skinny_fp8_half(int, int, long long);
extern "C" void qsa_skinny_fp8_block(int, int, long long, int, int, int*, int*);
extern "C" int qsa_skinny_gemm_fp8_probe_launch(
    const unsigned short*, const unsigned char*, const float*,
    unsigned short*, int, int, long long, long long, int, int, int,
    hipStream_t);
extern "C" void qsa_embed_rows_launch(const unsigned short*, const long long*,
                                      const unsigned short*, unsigned short*,
                                      unsigned short*, float*, int, int,
                                      long long, int, hipStream_t);
extern "C" void qsa_gemm_fp8_batch_launch(const unsigned short*,
                                          const unsigned char*,
                                          const float*, unsigned short*,
                                          float*, int, int, long long,
                                          long long, int, hipStream_t);
extern "C" void qsa_hash_build_launch(const long long*, const long long*,
                                      unsigned long long*, int, unsigned int,
                                      hipStream_t);
extern "C" void qsa_hash_probe_launch(const long long*,
                                      const unsigned long long*,
                                      const unsigned long long*, int*, int,
                                      unsigned int, long long, int,
                                      hipStream_t);
extern "C" bool qsa_short_gemm_takes(long long, long long, long long);
extern "C" void qsa_short_gemm_launch(const unsigned short*,
                                      const unsigned short*, unsigned short*,
                                      int, int, int, long long, int,
                                      hipStream_t);
extern "C" void qsa_encoder_attn_launch(
    const unsigned short*, const float*, const float*, int, const int*,
    const int*, const int*, const int*, unsigned short*, int, int, int, float,
    hipStream_t);
extern "C" int qsa_topk_block_docs(long long, long long);
extern "C" void qsa_topk_scan_launch(const float*, const float*, float*, int*,
                                     int, int, int, int, int, hipStream_t);
extern "C" void qsa_topk_fetch_launch(const float*, float*, long long,
                                      hipStream_t);
extern "C" int qsa_topk_groups(int);
extern "C" void qsa_topk_merge_launch(const float*, const int*, float*, int*,
                                      int, int, int, hipStream_t);
extern "C" void qsa_window_agg_launch(const long long*, const int*,
                                      const float*, int*, float*, long long,
                                      long long, int, int, long long, int*,
                                      hipStream_t);
extern "C" void qsa_window_clear_launch(int*, long long, hipStream_t);
extern "C" long long qsa_window_workspace(long long, long long, long long,
                                          long long);
void register_avro(pybind11::module_&);  // avro_codec.cpp
void register_bpe(pybind11::module_&);   // bpe.cpp
extern "C" void qsa_anomaly_batch_launch(const float*, const int*, float*,
                                         float*, int*, int, int, int,
                                         hipStream_t);

// ---------------------------------------------------------------------------

torch::Tensor rmsnorm(torch::Tensor x, torch::Tensor w, double eps) {
  CHK_DEV(x); CHK_CONT(x); CHK_BF16(x); CHK_BF16(w); CHK_CONT(w);
  const int H = x.size(-1);
  TORCH_CHECK(H % 8 == 0, "H % 8 == 0");
  const long long rows = x.numel() / H;
  auto y = torch::empty_like(x);
  qsa_rmsnorm_launch(u16(x), u16(w), u16m(y), nullptr, rows, H, (float)eps,
                     cur_stream());
  return y;
}

torch::Tensor rmsnorm_residual(torch::Tensor x, torch::Tensor res,
                               torch::Tensor w, double eps) {
  CHK_DEV(x); CHK_CONT(x); CHK_BF16(x); CHK_BF16(res); CHK_CONT(res);
  CHK_BF16(w); CHK_CONT(w);
  const int H = x.size(-1);
  TORCH_CHECK(H % 8 == 0, "H % 8 == 0");
  TORCH_CHECK(res.sizes() == x.sizes(), "residual shape mismatch");
  const long long rows = x.numel() / H;
  auto y = torch::empty_like(x);
  qsa_rmsnorm_launch(u16(x), u16(w), u16m(y), u16m(res), rows, H, (float)eps,
                     cur_stream());
  return y;
}

torch::Tensor swiglu(torch::Tensor gate, torch::Tensor up) {
  // gate/up: [rows, cols] views with equal row stride (e.g. halves of the
  // fused gate_up GEMM output); cols % 8 == 0, element-contiguous rows.
  CHK_DEV(gate); CHK_BF16(gate); CHK_BF16(up);
  TORCH_CHECK(gate.dim() == 2 && up.dim() == 2, "2-D");
  TORCH_CHECK(gate.sizes() == up.sizes(), "shape mismatch");
  TORCH_CHECK(gate.stride(1) == 1 && up.stride(1) == 1, "rows contiguous");
  TORCH_CHECK(gate.stride(0) == up.stride(0), "row strides must match");
  const long long rows = gate.size(0), cols = gate.size(1);
  TORCH_CHECK(cols % 8 == 0, "cols % 8 == 0");
  auto y = torch::empty({rows, cols}, gate.options());
  const long long n = rows * cols;
  const int blocks = (int)std::min<long long>((n / 8 + 255) / 256, 8192);
  qsa_swiglu_launch(u16(gate), u16(up), u16m(y), rows, cols, gate.stride(0),
                    blocks, cur_stream());
  return y;
}

static inline void chk_hd_strided(const torch::Tensor& t, int D,
                                  const char* name) {
  TORCH_CHECK(t.dim() == 3 && t.stride(2) == 1 && t.stride(1) == D,
              name, " must be a [B, H, D] view with contiguous heads");
}

void rope_inplace(torch::Tensor q, torch::Tensor k, torch::Tensor cos_t,
                  torch::Tensor sin_t, torch::Tensor pos) {
  CHK_DEV(q); CHK_BF16(q); CHK_BF16(k);
  CHK_F32(cos_t); CHK_F32(sin_t); CHK_I32(pos);
  const int B = q.size(0), QH = q.size(1), D = q.size(2);
  const int KVH = k.size(1);
  TORCH_CHECK(k.size(0) == B && k.size(2) == D, "k shape");
  chk_hd_strided(q, D, "q"); chk_hd_strided(k, D, "k");
  qsa_rope_launch(u16m(q), u16m(k), cos_t.data_ptr<float>(),
                  sin_t.data_ptr<float>(), pos.data_ptr<int>(), B, QH, KVH, D,
                  q.stride(0), k.stride(0), cur_stream());
}

void softmax_rows_(torch::Tensor scores, long col_offset, bool causal,
                   long row_mod, c10::optional<torch::Tensor> row_limits) {
  CHK_DEV(scores); CHK_CONT(scores); CHK_F32(scores);
  const int rows = scores.size(0), cols = scores.size(1);
  const int* rl = nullptr;
  if (row_limits.has_value()) {
    CHK_I32(row_limits.value());
    rl = row_limits.value().data_ptr<int>();
  }
  qsa_softmax_rows_launch(scores.data_ptr<float>(), rows, cols,
                          (int)col_offset, causal ? 1 : 0, (int)row_mod, rl,
                          cur_stream());
}

void softmax_rows_bf16_(torch::Tensor scores, double scale,
                        torch::Tensor row_limits) {
  CHK_DEV(scores); CHK_CONT(scores); CHK_BF16(scores); CHK_I32(row_limits);
  const long long rows = scores.size(0);
  const int cols = scores.size(1);
  TORCH_CHECK(cols % 8 == 0, "cols % 8 == 0");
  TORCH_CHECK(row_limits.numel() == rows, "one limit per row");
  qsa_softmax_rows_bf16_launch(u16m(scores), rows, cols, (float)scale,
                               row_limits.data_ptr<int>(), cur_stream());
}

// ---- activations of a decoding step ---------------------------------------
// Up to 4 rows are kept row-major [M, K], more of them packed in fragments
// [K/32, row tiles, 64, 8] (skinny_stream.h).
static int step_tiles(long M) { return M <= 4 ? 0 : M <= 16 ? 1 : 2; }

static torch::Tensor step_rows(long M, long K, torch::TensorOptions opts) {
  const int mt = step_tiles(M);
  return mt ? torch::empty({K / 32, mt, 64, 8}, opts)
            : torch::empty({M, K}, opts);
}

static torch::Tensor decode_attention(
    const torch::Tensor& q, const torch::Tensor* k, const torch::Tensor* v,
    torch::Tensor& kc, torch::Tensor& vc, const float* cos_t,
    const float* sin_t, const torch::Tensor& block_table,
    const torch::Tensor& seq_lens, double scale, bool step,
    const std::vector<torch::Tensor>& warm = {}) {
  CHK_DEV(q); CHK_BF16(q); CHK_BF16(kc); CHK_BF16(vc);
  CHK_CONT(kc); CHK_CONT(vc); CHK_I32(block_table); CHK_I32(seq_lens);
  CHK_CONT(block_table);
  const int B = q.size(0), QH = q.size(1), D = q.size(2);
  chk_hd_strided(q, D, "q");
  const int KVH = kc.size(1);
  TORCH_CHECK(D == 128 || D == 64, "D must be 64/128");
  TORCH_CHECK(QH % KVH == 0, "GQA requires QH % KVH == 0");
  TORCH_CHECK(QH / KVH <= 16, "GQA ratio <= 16");
  TORCH_CHECK(kc.size(2) == D / 8 && kc.size(3) == 64 && kc.size(4) == 8,
              "K cache layout [P, KVH, D/8, 64, 8]");
  TORCH_CHECK(vc.size(2) == D && vc.size(3) == 64,
              "V cache layout [P, KVH, D, 64] (transposed)");
  TORCH_CHECK(!step || (B >= 1 && B <= 32), "step rows: B in [1,32]");
  TORCH_CHECK(block_table.dim() == 2 && seq_lens.numel() >= B,
              "block_table [B, pages], a length per row");
  const int max_pages = block_table.size(1);
  const int mt = step ? step_tiles(B) : 0;
  auto out = mt ? step_rows(B, (long)QH * D, q.options())
                : torch::empty({B, QH, D}, q.options());
  // Every row's first page is read beside its length, so a table without pages
  // (all rows empty) and one without the last rows (these empty) have no launch
  // or get the rows.
  if (B == 0 || max_pages == 0) return out.zero_();
  const torch::Tensor table =
      block_table.size(0) >= B
          ? block_table
          : at::constant_pad_nd(block_table, {0, 0, 0, B - block_table.size(0)});
  int waves, ns;
  qsa_paged_attn_split(B, QH, KVH, max_pages, D, &waves, &ns);
  torch::Tensor part_o, part_ml;
  if (ns > 1) {
    auto opts_f = q.options().dtype(at::kFloat);
    part_o = torch::empty({B, QH, ns, D}, opts_f);
    part_ml = torch::empty({B, QH, ns, 2}, opts_f);
  }
  TORCH_CHECK(warm.size() <= 2, "at most two tensors to read ahead");
  const void* at[2] = {nullptr, nullptr};
  long long bytes[2] = {0, 0};
  for (size_t i = 0; i < warm.size(); ++i) {
    CHK_DEV(warm[i]); CHK_CONT(warm[i]);
    at[i] = warm[i].data_ptr();
    bytes[i] = reinterpret_cast<uintptr_t>(at[i]) & 15
        ? 0 : (long long)warm[i].nbytes();
  }
  qsa_paged_attn_mfma_launch(
      u16(q), k ? u16(*k) : nullptr, v ? u16(*v) : nullptr, u16m(kc), u16m(vc),
      cos_t, sin_t, table.data_ptr<int>(), seq_lens.data_ptr<int>(),
      ns > 1 ? part_o.data_ptr<float>() : nullptr,
      ns > 1 ? part_ml.data_ptr<float>() : nullptr, u16m(out), (float)scale, B,
      QH, KVH, max_pages, D, q.stride(0), k ? k->stride(0) : 0, waves, ns, mt,
      at, bytes, cur_stream());
  return out;
}

// (waves of a block, blocks per row and key head) that decode_attention takes
std::tuple<int, int> paged_attn_split(long B, long QH, long KVH,
                                      long max_pages, long D) {
  int waves, ns;
  qsa_paged_attn_split((int)B, (int)QH, (int)KVH, (int)max_pages, (int)D,
                       &waves, &ns);
  return {waves, ns};
}

torch::Tensor paged_attn_decode(torch::Tensor q, torch::Tensor kc,
                                torch::Tensor vc, torch::Tensor block_table,
                                torch::Tensor seq_lens, double scale) {
  return decode_attention(q, nullptr, nullptr, kc, vc, nullptr, nullptr,
                          block_table, seq_lens, scale, false);
}

torch::Tensor paged_attn_step(torch::Tensor q, torch::Tensor k,
                              torch::Tensor v, torch::Tensor kc,
                              torch::Tensor vc, torch::Tensor cos_t,
                              torch::Tensor sin_t, torch::Tensor block_table,
                              torch::Tensor seq_lens, double scale,
                              bool step, std::vector<torch::Tensor> warm) {
  // rope_kv_append and paged_attn_decode in one; q, k and v stay as they
  // are.  step: the result as step rows instead of [B, QH, D]
  CHK_BF16(k); CHK_BF16(v); CHK_F32(cos_t); CHK_F32(sin_t);
  CHK_CONT(cos_t); CHK_CONT(sin_t);
  const int D = q.size(2);
  chk_hd_strided(k, D, "k"); chk_hd_strided(v, D, "v");
  TORCH_CHECK(k.size(0) == q.size(0) && k.size(1) == kc.size(1) &&
                  v.sizes() == k.sizes(), "k/v [B, KVH, D]");
  TORCH_CHECK(k.stride(0) == v.stride(0), "k/v strides must match");
  TORCH_CHECK(q.stride(0) % 8 == 0 && k.stride(0) % 8 == 0 &&
                  ((reinterpret_cast<uintptr_t>(q.data_ptr()) |
                    reinterpret_cast<uintptr_t>(k.data_ptr())) & 15) == 0,
              "q and k rows must be 16-byte aligned");
  TORCH_CHECK(cos_t.size(-1) == D / 2 && sin_t.size(-1) == D / 2,
              "cos/sin [positions, D/2]");
  return decode_attention(q, &k, &v, kc, vc, cos_t.data_ptr<float>(),
                          sin_t.data_ptr<float>(), block_table, seq_lens,
                          scale, step, warm);
}

void kv_append(torch::Tensor knew, torch::Tensor vnew, torch::Tensor kc,
               torch::Tensor vc, torch::Tensor block_table,
               torch::Tensor seq_lens) {
  CHK_DEV(knew); CHK_BF16(knew); CHK_BF16(vnew);
  CHK_I32(block_table); CHK_I32(seq_lens);
  const int B = knew.size(0), KVH = knew.size(1), D = knew.size(2);
  chk_hd_strided(knew, D, "knew"); chk_hd_strided(vnew, D, "vnew");
  TORCH_CHECK(knew.stride(0) == vnew.stride(0), "k/v row strides must match");
  qsa_kv_append_launch(u16(knew), u16(vnew), u16m(kc), u16m(vc),
                       block_table.data_ptr<int>(), seq_lens.data_ptr<int>(),
                       B, KVH, D, (int)block_table.size(1), knew.stride(0),
                       cur_stream());
}

torch::Tensor paged_attn_prefill(torch::Tensor q, torch::Tensor kc,
                                 torch::Tensor vc, torch::Tensor block_table,
                                 torch::Tensor qb_item, torch::Tensor qb_pos0,
                                 torch::Tensor item_off,
                                 torch::Tensor item_start,
                                 torch::Tensor item_len, double scale,
                                 bool causal, long rows,
                                 c10::optional<torch::Tensor> cos_t,
                                 c10::optional<torch::Tensor> sin_t) {
  // rows: query tokens per block of the maps (qb_item, qb_pos0); with cos_t and
  // sin_t q is rotated here, by a row's position
  CHK_DEV(q); CHK_BF16(q); CHK_BF16(kc); CHK_BF16(vc);
  CHK_CONT(kc); CHK_CONT(vc); CHK_I32(block_table); CHK_CONT(block_table);
  CHK_I32(qb_item); CHK_I32(qb_pos0); CHK_I32(item_off);
  CHK_I32(item_start); CHK_I32(item_len);
  const int T = q.size(0), QH = q.size(1), D = q.size(2);
  chk_hd_strided(q, D, "q");
  const int KVH = kc.size(1);
  TORCH_CHECK(D == 128 || D == 64, "D must be 64/128");
  TORCH_CHECK(QH % KVH == 0 && QH / KVH <= 16, "GQA ratio <= 16");
  TORCH_CHECK(QH % 4 == 0, "QH % 4 == 0");
  TORCH_CHECK(rows >= 1 && rows <= 4096, "rows in [1,4096]");
  TORCH_CHECK(vc.size(2) == D && vc.size(3) == 64, "V layout [P,KVH,D,64]");
  const int QB = qb_item.numel();
  const int npmax = block_table.size(1);
  TORCH_CHECK(cos_t.has_value() == sin_t.has_value(), "cos and sin");
  if (cos_t) {
    CHK_F32(*cos_t); CHK_F32(*sin_t); CHK_CONT(*cos_t); CHK_CONT(*sin_t);
    TORCH_CHECK(cos_t->dim() == 2 && cos_t->size(1) == D / 2 &&
                    cos_t->size(0) > 0 && sin_t->sizes() == cos_t->sizes(),
                "cos/sin [positions, D/2]");
    TORCH_CHECK(cos_t->device() == q.device() && sin_t->device() == q.device(),
                "cos and sin must be where q is");
    TORCH_CHECK(((reinterpret_cast<uintptr_t>(cos_t->data_ptr()) |
                  reinterpret_cast<uintptr_t>(sin_t->data_ptr())) & 15) == 0,
                "cos and sin must be 16-byte aligned");
  }
  auto out = torch::empty({(long long)T, (long long)QH * D}, q.options());
  qsa_paged_attn_prefill_launch(
      u16(q), u16(kc), u16(vc), block_table.data_ptr<int>(),
      qb_item.data_ptr<int>(), qb_pos0.data_ptr<int>(),
      item_off.data_ptr<int>(), item_start.data_ptr<int>(),
      item_len.data_ptr<int>(), u16m(out), (float)scale, QB, QH, KVH, npmax,
      D, q.stride(0), causal ? 1 : 0, (int)rows,
      cos_t ? cos_t->data_ptr<float>() : nullptr,
      sin_t ? sin_t->data_ptr<float>() : nullptr,
      cos_t ? (int)cos_t->size(0) : 0, cur_stream());
  return out;
}

void rope_kv_append(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                    torch::Tensor kc, torch::Tensor vc, torch::Tensor cos_t,
                    torch::Tensor sin_t, torch::Tensor block_table,
                    torch::Tensor seq_lens) {
  CHK_DEV(q); CHK_BF16(q); CHK_BF16(k); CHK_BF16(v);
  CHK_F32(cos_t); CHK_F32(sin_t); CHK_I32(block_table); CHK_I32(seq_lens);
  CHK_CONT(block_table);
  const int B = q.size(0), QH = q.size(1), D = q.size(2);
  const int KVH = k.size(1);
  chk_hd_strided(q, D, "q"); chk_hd_strided(k, D, "k");
  chk_hd_strided(v, D, "v");
  TORCH_CHECK(k.stride(0) == v.stride(0), "k/v strides must match");
  qsa_rope_kv_append_launch(u16m(q), u16(k), u16(v), u16m(kc), u16m(vc),
                            cos_t.data_ptr<float>(), sin_t.data_ptr<float>(),
                            block_table.data_ptr<int>(),
                            seq_lens.data_ptr<int>(), B, QH, KVH, D,
                            (int)block_table.size(1), q.stride(0),
                            k.stride(0), cur_stream());
}

void rope_kv_scatter(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                     torch::Tensor kc, torch::Tensor vc, torch::Tensor cos_t,
                     torch::Tensor sin_t, torch::Tensor pos,
                     torch::Tensor slots, bool turn_q) {
  // rope_inplace on q (unless its reader turns it), and k rotated and v written to
  // the pages; k and v stay
  CHK_DEV(q); CHK_BF16(q); CHK_BF16(k); CHK_BF16(v);
  CHK_BF16(kc); CHK_BF16(vc); CHK_CONT(kc); CHK_CONT(vc);
  CHK_F32(cos_t); CHK_F32(sin_t); CHK_CONT(cos_t); CHK_CONT(sin_t);
  CHK_I32(pos); CHK_I32(slots); CHK_CONT(pos); CHK_CONT(slots);
  const int T = q.size(0), QH = q.size(1), D = q.size(2);
  const int KVH = k.size(1);
  TORCH_CHECK(D == 128 || D == 64, "D must be 64/128");
  TORCH_CHECK(QH % KVH == 0, "GQA requires QH % KVH == 0");
  TORCH_CHECK(k.size(0) == T && k.size(2) == D && v.sizes() == k.sizes() &&
                  pos.numel() == T && slots.numel() == T, "k/v/pos/slots [T]");
  TORCH_CHECK(kc.dim() == 5 && kc.size(1) == KVH && kc.size(2) == D / 8 &&
                  kc.size(3) == 64 && kc.size(4) == 8 && vc.dim() == 4 &&
                  vc.size(1) == KVH && vc.size(2) == D && vc.size(3) == 64,
              "cache layouts [P, KVH, D/8, 64, 8], [P, KVH, D, 64]");
  TORCH_CHECK(cos_t.size(-1) == D / 2 && sin_t.size(-1) == D / 2,
              "cos/sin [positions, D/2]");
  chk_hd_strided(q, D, "q"); chk_hd_strided(k, D, "k");
  chk_hd_strided(v, D, "v");
  TORCH_CHECK(k.stride(0) == v.stride(0), "k/v strides must match");
  TORCH_CHECK(q.stride(0) % 8 == 0 && k.stride(0) % 8 == 0 &&
                  ((reinterpret_cast<uintptr_t>(q.data_ptr()) |
                    reinterpret_cast<uintptr_t>(k.data_ptr()) |
                    reinterpret_cast<uintptr_t>(v.data_ptr())) & 15) == 0,
              "q, k and v rows must be 16-byte aligned");
  if (T == 0) return;
  qsa_rope_kv_scatter_launch(u16m(q), u16(k), u16(v), u16m(kc), u16m(vc),
                             cos_t.data_ptr<float>(), sin_t.data_ptr<float>(),
                             pos.data_ptr<int>(), slots.data_ptr<int>(), T,
                             turn_q ? QH : 0, KVH, D, q.stride(0), k.stride(0), cur_stream());
}

torch::Tensor mean_rows(torch::Tensor x, torch::Tensor off,
                        torch::Tensor len) {
  CHK_DEV(x); CHK_BF16(x); CHK_CONT(x); CHK_I32(off); CHK_I32(len);
  CHK_CONT(off); CHK_CONT(len);
  TORCH_CHECK(x.dim() == 2 && x.size(1) % 8 == 0, "x [T, H], H % 8 == 0");
  TORCH_CHECK(off.numel() == len.numel(), "off and len per item");
  const int n = off.numel(), H = x.size(1);
  auto out = torch::empty({n, H}, x.options().dtype(at::kFloat));
  if (n)
    qsa_mean_rows_launch(u16(x), off.data_ptr<int>(), len.data_ptr<int>(),
                         out.data_ptr<float>(), n, H, cur_stream());
  return out;
}

void kv_scatter(torch::Tensor knew, torch::Tensor vnew, torch::Tensor kc,
                torch::Tensor vc, torch::Tensor slots) {
  CHK_DEV(knew); CHK_BF16(knew); CHK_BF16(vnew); CHK_I32(slots);
  const int T = knew.size(0), KVH = knew.size(1), D = knew.size(2);
  chk_hd_strided(knew, D, "knew"); chk_hd_strided(vnew, D, "vnew");
  TORCH_CHECK(knew.stride(0) == vnew.stride(0), "k/v strides must match");
  if (T == 0) return;
  qsa_kv_scatter_launch(u16(knew), u16(vnew), u16m(kc), u16m(vc),
                        slots.data_ptr<int>(), T, KVH, D, knew.stride(0),
                        cur_stream());
}

torch::Tensor pack_weight_frag(torch::Tensor w) {
  // [N, K] bf16 -> MFMA-fragment-major [N/16, K/32, 16, 32] for the
  // skinny-GEMM weight stream (one wave reads one contiguous 1 KiB block).
  CHK_BF16(w); CHK_CONT(w);
  const long long N = w.size(0), K = w.size(1);
  TORCH_CHECK(N % 16 == 0 && K % 32 == 0, "pack needs N%16==0, K%32==0");
  return w.reshape({N / 16, 16, K / 32, 32})
      .permute({0, 2, 1, 3}).contiguous();
}

// What the weight streams (skinny_stream.h) read by descriptors of 32-bit offsets, in
// whole 16 bytes: a copy where a tensor does not start on one, or its rows are not that
// or too far apart.
static torch::Tensor whole16(torch::Tensor t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) & 15
             ? t.clone(at::MemoryFormat::Contiguous) : t;
}
static torch::Tensor stream_rows(torch::Tensor a) {
  return a.stride(0) % 8 || a.size(0) * a.stride(0) >= 1ll << 30
             ? a.clone(at::MemoryFormat::Contiguous) : whole16(a);
}

torch::Tensor skinny_gemm(torch::Tensor a, torch::Tensor wf, long N, long K) {
  // C[M,N] = a[M,K] @ W^T with W pre-packed by pack_weight_frag.
  CHK_DEV(a); CHK_BF16(a); CHK_BF16(wf); CHK_CONT(wf);
  TORCH_CHECK(a.dim() == 2 && a.stride(1) == 1, "a rows must be contiguous");
  const int M = a.size(0);
  TORCH_CHECK(M >= 1 && M <= 32, "skinny_gemm: M in [1,32]");
  TORCH_CHECK(a.size(1) == K, "K mismatch");
  TORCH_CHECK(K % 256 == 0 && N % 16 == 0, "K%256==0, N%16==0");
  TORCH_CHECK(wf.numel() == (long long)N * K, "wf size");
  a = stream_rows(a);
  wf = whole16(wf);
  auto out = torch::empty({M, (long long)N}, a.options());
  qsa_skinny_gemm_launch(u16(a), u16(wf), u16m(out), M, (int)N, K,
                         a.stride(0), false, cur_stream());
  return out;
}

torch::Tensor skinny_gemm_probe(torch::Tensor a, torch::Tensor wf, long N,
                                long K, long waves, long tiles) {
  CHK_DEV(a); CHK_BF16(a); CHK_BF16(wf); CHK_CONT(wf);
  const int M = a.size(0);
  TORCH_CHECK(M >= 1 && M <= 32 && N % (16 * tiles) == 0 && K % 64 == 0 &&
                  wf.numel() == (long long)N * K && a.size(1) == K,
              "skinny_gemm_probe: shapes");
  a = stream_rows(a);
  wf = whole16(wf);
  auto out = torch::empty({M, (long long)N}, a.options());
  TORCH_CHECK(qsa_skinny_gemm_probe_launch(u16(a), u16(wf), u16m(out), M,
                                           (int)N, K, a.stride(0), (int)waves,
                                           (int)tiles, cur_stream()),
              "skinny_gemm_probe: no such block shape");
  return out;
}

torch::Tensor gemm_fp8_batch(torch::Tensor a, torch::Tensor qf,
                             torch::Tensor scale, long N, long K,
                             long splitk) {
  // C[M,N] = a @ (scale * dequant(Q))^T for decode batches 32 < M <= 256
  CHK_DEV(a); CHK_BF16(a); CHK_CONT(qf);
  TORCH_CHECK(qf.scalar_type() == torch::kUInt8, "qf must be uint8 (fp8)");
  TORCH_CHECK(scale.scalar_type() == torch::kFloat32 && scale.is_cuda() &&
                  scale.is_contiguous() && scale.numel() == N, "scale");
  TORCH_CHECK(a.dim() == 2 && a.stride(1) == 1, "a rows must be contiguous");
  const int M = a.size(0);
  TORCH_CHECK(M >= 1 && M <= 256, "gemm_fp8_batch: M in [1,256]");
  TORCH_CHECK(a.size(1) == K, "K mismatch");
  TORCH_CHECK(N % 64 == 0, "N % 64 == 0");
  TORCH_CHECK(splitk == 1 || splitk == 2 || splitk == 4, "splitk 1/2/4");
  TORCH_CHECK(K % (64 * splitk) == 0, "K % (64*splitk) == 0");
  TORCH_CHECK(qf.numel() == (long long)N * K, "qf size");
  auto out = torch::empty({(long long)M, (long long)N}, a.options());
  torch::Tensor ws;
  float* wsp = nullptr;
  if (splitk > 1) {
    ws = torch::empty({splitk, (long long)M, (long long)N},
                      a.options().dtype(torch::kFloat32));
    wsp = ws.data_ptr<float>();
  }
  qsa_gemm_fp8_batch_launch(u16(a), qf.data_ptr<unsigned char>(),
                            scale.data_ptr<float>(), u16m(out), wsp, M,
                            (int)N, K, a.stride(0), (int)splitk,
                            cur_stream());
  return out;
}

std::vector<torch::Tensor> hash_build(torch::Tensor keys,
                                      torch::Tensor ts) {
  // latest-event-time-per-key hash table in HBM (K8 streaming join state)
  CHK_DEV(keys);
  TORCH_CHECK(keys.scalar_type() == torch::kInt64 && keys.is_contiguous(),
              "keys must be contiguous i64");
  TORCH_CHECK(ts.scalar_type() == torch::kInt64 && ts.is_contiguous() &&
                  ts.numel() == keys.numel(), "ts must be i64 like keys");
  const long long n = keys.numel();
  TORCH_CHECK(n < (1 << 24), "hash_build: <= 2^24 rows per batch");
  long long cap = 64;
  while (cap < 2 * n) cap <<= 1;
  // slots of (key, payload) pairs, handed out as two strided views
  auto slots = torch::empty({cap, 2}, keys.options());
  qsa_hash_build_launch((const long long*)keys.data_ptr<int64_t>(),
                        (const long long*)ts.data_ptr<int64_t>(),
                        (unsigned long long*)slots.data_ptr<int64_t>(),
                        (int)n, (unsigned int)(cap - 1), cur_stream());
  return {slots.select(1, 0), slots.select(1, 1)};
}

torch::Tensor hash_probe(torch::Tensor tkeys, torch::Tensor tpay,
                         torch::Tensor keys, long long min_ts) {
  CHK_DEV(keys);
  TORCH_CHECK(keys.scalar_type() == torch::kInt64 && keys.is_contiguous(),
              "keys must be contiguous i64");
  const long long m = keys.numel();
  const long long cap = tkeys.numel();
  TORCH_CHECK((cap & (cap - 1)) == 0, "table capacity must be pow2");
  auto out = torch::empty({m}, keys.options().dtype(torch::kInt32));
  const int64_t* words = tkeys.data_ptr<int64_t>();
  const bool paired = tkeys.stride(0) == 2 && tpay.stride(0) == 2 &&
                      tpay.data_ptr<int64_t>() == words + 1 &&
                      (reinterpret_cast<uintptr_t>(words) & 15) == 0;
  if (!paired) {
    tkeys = tkeys.contiguous();
    tpay = tpay.contiguous();
  }
  qsa_hash_probe_launch((const long long*)keys.data_ptr<int64_t>(),
                        (const unsigned long long*)tkeys.data_ptr<int64_t>(),
                        (const unsigned long long*)tpay.data_ptr<int64_t>(),
                        out.data_ptr<int>(), (int)m,
                        (unsigned int)(cap - 1), min_ts, paired,
                        cur_stream());
  return out;
}

static void chk_fp8_weight(const torch::Tensor& qf, const torch::Tensor& scale,
                           long N, long K) {
  CHK_DEV(qf); CHK_CONT(qf);
  TORCH_CHECK(qf.scalar_type() == torch::kUInt8, "qf must be uint8 (fp8)");
  TORCH_CHECK(scale.scalar_type() == torch::kFloat32 && scale.is_cuda() &&
                  scale.is_contiguous() && scale.numel() == N,
              "scale must be f32 [N] on device");
  TORCH_CHECK(K % 256 == 0 && N % 16 == 0, "K%256==0, N%16==0");
  TORCH_CHECK(qf.numel() == (long long)N * K, "qf size");
}

static int chk_skinny_fp8(const torch::Tensor& a, const torch::Tensor& qf,
                          const torch::Tensor& scale, long N, long K) {
  CHK_DEV(a); CHK_BF16(a);
  TORCH_CHECK(a.dim() == 2 && a.stride(1) == 1, "a rows must be contiguous");
  const int M = a.size(0);
  TORCH_CHECK(M >= 1 && M <= 32, "skinny_gemm_fp8: M in [1,32]");
  TORCH_CHECK(a.size(1) == K, "K mismatch");
  chk_fp8_weight(qf, scale, N, K);
  return M;
}

torch::Tensor skinny_gemm_fp8(torch::Tensor a, torch::Tensor qf,
                              torch::Tensor scale, long N, long K, bool far) {
  // C[M,N] = a @ (scale[N] * dequant(Q))^T; Q pre-packed fp8 e4m3 in the
  // fragment-pair-major stream layout (skinny_gemm_fp8.hip header).
  const int M = chk_skinny_fp8(a, qf, scale, N, K);
  a = stream_rows(a);
  qf = whole16(qf);
  auto out = torch::empty({M, (long long)N}, a.options());
  qsa_skinny_gemm_fp8_launch(u16(a), qf.data_ptr<unsigned char>(),
                             scale.data_ptr<float>(), u16m(out), nullptr, M,
                             (int)N, K, a.stride(0), 0, nullptr, nullptr, 0,
                             0.f, 0, nullptr, far, cur_stream());
  return out;
}

// step rows, their sums of squares being [32, parts4] (parts rounded up to 4)
static void chk_step_rows(const torch::Tensor& a, long M, long K) {
  CHK_DEV(a); CHK_BF16(a); CHK_CONT(a);
  TORCH_CHECK(M >= 1 && M <= 32, "step rows: M in [1,32]");
  const int mt = step_tiles(M);
  TORCH_CHECK(mt ? a.dim() == 4 && a.size(1) == mt &&
                       a.numel() == (long long)K * mt * 16
                 : a.dim() == 2 && a.size(0) == M && a.size(1) == K,
              "step rows: shape");
}

torch::Tensor skinny_gemm_fp8_norm(torch::Tensor a, torch::Tensor ss,
                                   long parts, long M, double eps,
                                   torch::Tensor qf, torch::Tensor scale,
                                   long N, long K, bool glu, bool far) {
  // a: rows x * w of an rms norm; 1/rms from the rows' sums of squares.
  // glu: Q's rows are [gate; up], returns silu(gate) * up as step rows.
  chk_step_rows(a, M, K);
  chk_fp8_weight(qf, scale, N, K);
  CHK_DEV(ss); CHK_F32(ss); CHK_CONT(ss);
  TORCH_CHECK(parts >= 1 && ss.numel() == 32 * ((parts + 3) & ~3L),
              "sums of squares [32, parts4]");
  TORCH_CHECK(!glu || N % 64 == 0, "gate and up: N % 64 == 0");
  a = whole16(a);
  qf = whole16(qf);
  auto out = glu ? step_rows(M, N / 2, a.options())
                 : torch::empty({(long long)M, (long long)N}, a.options());
  qsa_skinny_gemm_fp8_launch(u16(a), qf.data_ptr<unsigned char>(),
                             scale.data_ptr<float>(), u16m(out), nullptr,
                             (int)M, (int)N, K, K, step_tiles(M) > 0, nullptr,
                             ss.data_ptr<float>(), (int)parts, (float)eps,
                             glu ? 1 : 0, nullptr, far, cur_stream());
  return out;
}

// parts that skinny_gemm_fp8_residual leaves of a row's sum of squares
long skinny_gemm_fp8_parts(long M, long N, long K) {
  return N / (qsa_skinny_fp8_half((int)M, (int)N, K) ? 8 : 16);
}

// (waves, tiles of 16 columns) of a block
std::tuple<int, int> skinny_gemm_fp8_block(long M, long N, long K, bool glu,
                                           bool res) {
  int waves, tiles;
  qsa_skinny_fp8_block((int)M, (int)N, K, glu, res, &waves, &tiles);
  return {waves, tiles};
}

std::vector<torch::Tensor> skinny_gemm_fp8_residual(
    torch::Tensor a, torch::Tensor qf, torch::Tensor scale, long N, long K,
    torch::Tensor res, torch::Tensor w, bool far) {
  // res [M, N] <- res + the product; returns the rows of the norm with weight
  // w that follows (before 1/rms) and the sums of squares in their parts
  CHK_DEV(res); CHK_BF16(res); CHK_CONT(res);
  TORCH_CHECK(res.dim() == 2 && res.size(1) == N, "residual [M, N]");
  const long M = res.size(0);
  chk_step_rows(a, M, K);
  chk_fp8_weight(qf, scale, N, K);
  CHK_DEV(w); CHK_BF16(w); CHK_CONT(w);
  TORCH_CHECK(w.numel() == N && N % 32 == 0, "norm weight [N], N % 32 == 0");
  a = whole16(a);
  qf = whole16(qf);
  auto next = step_rows(M, N, a.options());
  auto ss = torch::empty({32, (skinny_gemm_fp8_parts(M, N, K) + 3) & ~3L},
                         a.options().dtype(at::kFloat));
  qsa_skinny_gemm_fp8_launch(u16(a), qf.data_ptr<unsigned char>(),
                             scale.data_ptr<float>(), u16m(res), u16m(next),
                             (int)M, (int)N, K, K, step_tiles(M) > 0, u16(w),
                             nullptr, 0, 0.f, 0, ss.data_ptr<float>(), far,
                             cur_stream());
  return {next, ss};
}

std::vector<torch::Tensor> embed_rows(torch::Tensor embed,
                                      torch::Tensor tokens,
                                      torch::Tensor w) {
  // (embed[tokens], the rows of the norm with weight w that follows, the
  // sums of squares in one part)
  CHK_DEV(embed); CHK_BF16(embed); CHK_CONT(embed); CHK_DEV(tokens);
  TORCH_CHECK((tokens.scalar_type() == torch::kInt64 ||
               tokens.scalar_type() == torch::kInt32) && tokens.dim() == 1,
              "tokens must be i64 or i32 [M]");
  // as index_select takes them; the engine's are i64 and contiguous
  tokens = tokens.to(torch::kInt64).contiguous();
  const long M = tokens.size(0), H = embed.size(1);
  TORCH_CHECK(M >= 1 && M <= 32 && H % 32 == 0, "M in [1,32], H % 32 == 0");
  CHK_DEV(w); CHK_BF16(w); CHK_CONT(w);
  TORCH_CHECK(w.numel() == H, "norm weight [H]");
  auto res = torch::empty({M, H}, embed.options());
  auto next = step_rows(M, H, embed.options());
  auto ss = torch::empty({32, 4}, embed.options().dtype(at::kFloat));
  qsa_embed_rows_launch(u16(embed),
                        (const long long*)tokens.data_ptr<int64_t>(), u16(w),
                        u16m(res), u16m(next), ss.data_ptr<float>(), (int)M,
                        (int)H, embed.size(0), step_tiles(M), cur_stream());
  return {res, next, ss};
}

torch::Tensor skinny_gemm_fp8_probe(torch::Tensor a, torch::Tensor qf,
                                    torch::Tensor scale, long M, long N,
                                    long K, long waves, long tiles) {
  // a: [M, K], or packed fragments
  chk_fp8_weight(qf, scale, N, K);
  CHK_DEV(a); CHK_BF16(a); CHK_CONT(a);
  const bool pack = a.dim() == 4;
  TORCH_CHECK(M >= 1 && M <= 32 && N % (16 * tiles) == 0 &&
                  a.numel() == (pack ? (M <= 16 ? 16 : 32) : M) * (long long)K,
              "skinny_gemm_fp8_probe: shapes");
  a = whole16(a);
  qf = whole16(qf);
  auto out = torch::empty({(long long)M, (long long)N}, a.options());
  TORCH_CHECK(qsa_skinny_gemm_fp8_probe_launch(
                  u16(a), qf.data_ptr<unsigned char>(),
                  scale.data_ptr<float>(), u16m(out), (int)M, (int)N, K, K,
                  pack, (int)waves, (int)tiles, cur_stream()),
              "skinny_gemm_fp8_probe: no such block shape");
  return out;
}

// a @ w^T, or with glu, w = [gate; up], silu(gate) * up of it
torch::Tensor short_gemm(torch::Tensor a, torch::Tensor w, bool glu) {
  CHK_DEV(a); CHK_DEV(w); CHK_BF16(a); CHK_BF16(w); CHK_CONT(w);
  TORCH_CHECK(a.dim() == 2 && w.dim() == 2 && a.stride(1) == 1 &&
                  a.size(1) == w.size(1), "a [M, K], w [N, K]");
  const long long M = a.size(0), N = w.size(0), K = w.size(1);
  TORCH_CHECK(K >= 64 && K % 64 == 0 && N >= 32 && N % (glu ? 32 : 16) == 0,
              "K % 64, N % 16");
  TORCH_CHECK(M < (1 << 24) && N < (1 << 20) && a.stride(0) % 8 == 0 &&
                  ((reinterpret_cast<uintptr_t>(a.data_ptr()) |
                    reinterpret_cast<uintptr_t>(w.data_ptr())) & 15) == 0,
              "sizes, alignment");
  auto out = torch::empty({M, glu ? N / 2 : N}, a.options());
  qsa_short_gemm_launch(u16(a), u16(w), u16m(out), (int)M, (int)N, (int)K,
                        a.stride(0), glu, cur_stream());
  return out;
}

// rows of [q | k | v] of the items, blocks of 64 query rows -> [T, H*D]
torch::Tensor encoder_attn(torch::Tensor qkv, torch::Tensor cos_t,
                           torch::Tensor sin_t, torch::Tensor qb_item,
                           torch::Tensor qb_t0, torch::Tensor off,
                           torch::Tensor len, long heads, double scale) {
  CHK_DEV(qkv); CHK_BF16(qkv); CHK_CONT(qkv);
  CHK_F32(cos_t); CHK_F32(sin_t); CHK_CONT(cos_t); CHK_CONT(sin_t);
  CHK_I32(qb_item); CHK_I32(qb_t0); CHK_I32(off); CHK_I32(len);
  TORCH_CHECK(qkv.dim() == 2 && heads > 0 && heads % 4 == 0 &&
                  qkv.size(1) % (3 * heads) == 0, "[T, 3 * heads * D]");
  const long long A = qkv.size(1) / 3, D = A / heads;
  TORCH_CHECK(D == 128 || D == 64, "D must be 64/128");
  TORCH_CHECK((reinterpret_cast<uintptr_t>(qkv.data_ptr()) & 15) == 0,
              "rows must be 16-byte aligned");
  TORCH_CHECK(cos_t.dim() == 2 && cos_t.size(0) >= 1 &&
                  cos_t.size(1) == D / 2 && sin_t.sizes() == cos_t.sizes(),
              "cos/sin [positions, D/2]");
  TORCH_CHECK(qb_item.numel() == qb_t0.numel() && off.numel() == len.numel(),
              "maps");
  auto out = torch::empty({qkv.size(0), A}, qkv.options());
  qsa_encoder_attn_launch(
      u16(qkv), cos_t.data_ptr<float>(), sin_t.data_ptr<float>(),
      (int)cos_t.size(0), qb_item.data_ptr<int>(), qb_t0.data_ptr<int>(),
      off.data_ptr<int>(), len.data_ptr<int>(), u16m(out),
      (int)qb_item.numel(), (int)heads, (int)D, (float)scale, cur_stream());
  return out;
}

// Scans and merges on the current stream.  The result is [2, Q, k]: scores, as the
// bits of floats, and documents, in `out` or, without it, in a tensor of its own.
static torch::Tensor topk_run(const torch::Tensor& queries,
                              const torch::Tensor& docs, long k, int* out) {
  const int Q = queries.size(0), D = queries.size(1), N = docs.size(0);
  TORCH_CHECK(docs.size(1) == D, "dim mismatch");
  TORCH_CHECK(k >= 1 && k <= 16, "k in [1,16]");
  const int per = qsa_topk_block_docs(Q, N);
  int lists = (N + per - 1) / per;
  const auto opt = queries.options().dtype(at::kInt);
  if (Q == 0) return torch::empty({2, 0, k}, opt);
  torch::Tensor kept, from;            // the candidates, and what they merge into
  auto lists_of = [&](long n) {
    if (n == 1 && out) return out;
    kept = torch::empty({2, Q, n * k}, opt);
    return kept.data_ptr<int>();
  };
  auto scores = [](int* at) { return reinterpret_cast<float*>(at); };
  auto ids = [&](int* at, long n) { return at + Q * n * k; };
  int* now = lists_of(lists);
  qsa_topk_scan_launch(queries.data_ptr<float>(), docs.data_ptr<float>(),
                       scores(now), ids(now, lists), Q, N, D, (int)k, lists,
                       cur_stream());
  // a single list is the result (5 rows, k = 5: 17.5 us with the merge)
  while (lists != 1) {
    const int groups = qsa_topk_groups(lists);
    from = kept;
    int* to = lists_of(groups);
    qsa_topk_merge_launch(scores(now), ids(now, lists), scores(to),
                          ids(to, groups), Q, lists, (int)k, cur_stream());
    now = to;
    lists = groups;
  }
  return kept;
}

torch::Tensor topk_cosine_packed(torch::Tensor queries, torch::Tensor docs,
                                 long k) {
  CHK_DEV(queries); CHK_CONT(queries); CHK_F32(queries); CHK_F32(docs);
  CHK_CONT(docs);
  return topk_run(queries, docs, k, nullptr);
}

// The same of queries on the host, normalized on the way, with the result on the
// host: array [2, Q, k], or none if a query holds what is not a number or infinite.
// Queries and result pass through pinned memory that a kernel reads and the last
// one writes, so that neither waits for a copy (see the caller for times).
py::object topk_cosine_host(
    py::array_t<float, py::array::c_style | py::array::forcecast> queries,
    torch::Tensor docs, long k) {
  CHK_DEV(docs); CHK_F32(docs); CHK_CONT(docs);
  TORCH_CHECK(queries.ndim() == 2, "queries must be rows");
  const long Q = queries.shape(0), D = queries.shape(1), n = Q * D;
  TORCH_CHECK(docs.dim() == 2 && docs.size(1) == D, "dim mismatch");
  TORCH_CHECK(k >= 1 && k <= 16, "k in [1,16]");
  py::array_t<int> result({2L, Q, k});
  if (Q == 0) return result;
  const float* q = queries.data();
  int* res = result.mutable_data();
  bool numbers = true;
  {
    py::gil_scoped_release release;
    const c10::DeviceGuard guard(docs.device());
    const long rows = (n + 3) / 4 * 4;
    auto pinned = torch::empty(
        {rows + 2 * Q * k},
        torch::TensorOptions().dtype(at::kFloat).pinned_memory(true));
    float* host = pinned.data_ptr<float>();
    for (long i = 0; i < Q && numbers; ++i) {
      double s[4] = {0, 0, 0, 0};      // four sums: vector operations
      const float* x = q + i * D;
      long j = 0;
      for (; j + 4 <= D; j += 4)
        for (int e = 0; e < 4; ++e) s[e] += (double)x[j + e] * x[j + e];
      for (; j < D; ++j) s[0] += (double)x[j] * x[j];
      const double sum = s[0] + s[1] + s[2] + s[3];
      numbers = std::isfinite(sum);    // squares of floats stay in range
      // rounded once, at the end; a norm beyond what floats hold is infinite
      const double inv = std::isinf((float)sum)
          ? 0.0 : 1.0 / std::max(std::sqrt(sum), 1e-12);
      for (j = 0; j < D; ++j) host[i * D + j] = (float)(x[j] * inv);
    }
    if (numbers) {
      auto rows_on = torch::empty({Q, D}, docs.options());
      qsa_topk_fetch_launch(host, rows_on.data_ptr<float>(), n, cur_stream());
      int* out = reinterpret_cast<int*>(host + rows);
      topk_run(rows_on, docs, k, out);
      // waits, and reports what the launches left
      const hipError_t err = hipStreamSynchronize(cur_stream());
      TORCH_CHECK(err == hipSuccess, "top-k search: ", hipGetErrorString(err));
      std::copy(out, out + 2 * Q * k, res);
    }
  }
  if (!numbers) return py::none();
  return result;
}

std::vector<torch::Tensor> topk_cosine(torch::Tensor queries,
                                       torch::Tensor docs, long k) {
  auto both = topk_cosine_packed(queries, docs, k);
  return {both[0].view(at::kFloat), both[1]};
}

std::vector<torch::Tensor> window_agg(torch::Tensor ts, torch::Tensor key,
                                      c10::optional<torch::Tensor> value,
                                      long t0, long win_ms, long nwin,
                                      long nkeys) {
  CHK_DEV(ts); CHK_CONT(ts); CHK_I32(key);
  TORCH_CHECK(ts.scalar_type() == at::kLong, "ts must be i64");
  const long long n = ts.numel();
  // one buffer: the two tables are cleared by one launch
  auto cells = torch::empty({2, nkeys, nwin}, key.options());
  qsa_window_clear_launch(cells.data_ptr<int>(), cells.numel(), cur_stream());
  auto counts = cells[0];
  auto sums = cells[1].view(at::kFloat);
  const float* vptr = nullptr;
  if (value.has_value()) {
    CHK_F32(value.value());
    vptr = value.value().data_ptr<float>();
  }
  const long long words = qsa_window_workspace(n, nkeys, nwin, win_ms);
  torch::Tensor ws;
  int* wptr = nullptr;
  if (words) {
    ws = torch::empty({words}, key.options());
    wptr = ws.data_ptr<int>();
  }
  qsa_window_agg_launch(reinterpret_cast<const long long*>(ts.data_ptr<int64_t>()),
                        key.data_ptr<int>(), vptr,
                        counts.data_ptr<int>(), sums.data_ptr<float>(), t0,
                        win_ms, (int)nwin, (int)nkeys, n, wptr,
                        cur_stream());
  return {counts, sums};
}

std::vector<torch::Tensor> anomaly_batch(torch::Tensor series,
                                         torch::Tensor lengths, long order) {
  CHK_DEV(series); CHK_CONT(series); CHK_F32(series); CHK_I32(lengths);
  const int K = series.size(0), Tmax = series.size(1);
  auto fc = torch::empty({K}, series.options());
  auto se = torch::empty({K}, series.options());
  auto dof = torch::empty({K}, series.options().dtype(at::kInt));
  qsa_anomaly_batch_launch(series.data_ptr<float>(), lengths.data_ptr<int>(),
                           fc.data_ptr<float>(), se.data_ptr<float>(),
                           dof.data_ptr<int>(), K, Tmax, (int)order,
                           cur_stream());
  return {fc, se, dof};
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rmsnorm", &rmsnorm, "fused RMSNorm (bf16)");
  m.def("rmsnorm_residual", &rmsnorm_residual,
        "fused residual-add + RMSNorm (bf16; residual updated in place)");
  m.def("swiglu", &swiglu, "fused silu(gate)*up (bf16)");
  m.def("rope_inplace", &rope_inplace, "rotary embedding in place (bf16)");
  m.def("softmax_rows_bf16_", &softmax_rows_bf16_,
        "bf16 masked row softmax with folded scale (in place)");
  m.def("softmax_rows_", &softmax_rows_, "row softmax in place (f32)",
        py::arg("scores"), py::arg("col_offset") = 0, py::arg("causal") = false,
        py::arg("row_mod") = 0, py::arg("row_limits") = py::none());
  m.def("paged_attn_prefill", &paged_attn_prefill,
        "varlen flash prefill attention over the paged cache",
        py::arg("q"), py::arg("kc"), py::arg("vc"), py::arg("block_table"),
        py::arg("qb_item"), py::arg("qb_pos0"), py::arg("item_off"),
        py::arg("item_start"), py::arg("item_len"), py::arg("scale"),
        py::arg("causal"), py::arg("rows") = 16, py::arg("cos_t") = py::none(),
        py::arg("sin_t") = py::none());
  m.def("paged_attn_decode", &paged_attn_decode,
        "paged-attention decode (bf16, GQA, page=64)");
  m.def("paged_attn_split", &paged_attn_split,
        "waves and blocks of a decoding step's attention");
  m.def("paged_attn_step", &paged_attn_step,
        "a decoding step's rotation, cache append and attention",
        py::arg("q"), py::arg("k"), py::arg("v"), py::arg("kc"),
        py::arg("vc"), py::arg("cos"), py::arg("sin"), py::arg("block_table"),
        py::arg("seq_lens"), py::arg("scale"), py::arg("step"),
        py::arg("warm") = std::vector<torch::Tensor>());
  m.def("kv_append", &kv_append, "append one step's k/v to the paged cache");
  m.def("rope_kv_append", &rope_kv_append,
        "fused decode rope + paged-cache append");
  m.def("rope_kv_scatter", &rope_kv_scatter,
        "prefill rotation and paged-cache write", py::arg("q"), py::arg("k"),
        py::arg("v"), py::arg("kc"), py::arg("vc"), py::arg("cos_t"),
        py::arg("sin_t"), py::arg("pos"), py::arg("slots"),
        py::arg("turn_q") = true);
  m.def("encoder_attn", &encoder_attn,
        "rotation and bidirectional attention of projection rows");
  m.def("short_gemm", &short_gemm, "GEMM of a short K, optionally gated");
  m.def("short_gemm_takes", &qsa_short_gemm_takes,
        "whether the encoder's product [M, N, K] is short_gemm's");
  m.def("mean_rows", &mean_rows, "mean of each item's rows (f32)");
  m.def("kv_scatter", &kv_scatter, "scatter prefill k/v by slot ids");
  m.def("pack_weight_frag", &pack_weight_frag,
        "repack [N,K] bf16 into MFMA-fragment-major for skinny_gemm");
  m.def("skinny_gemm", &skinny_gemm,
        "decode-batch GEMM (M<=32) on the packed weight stream");
  m.def("skinny_gemm_probe", &skinny_gemm_probe,
        "tuning probe: waves, tiles");
  m.def("skinny_gemm_fp8", &skinny_gemm_fp8,
        "fp8-weight decode GEMM (M<=32): half the weight stream",
        py::arg("a"), py::arg("qf"), py::arg("scale"), py::arg("N"),
        py::arg("K"), py::arg("far") = false);
  m.def("gemm_fp8_batch", &gemm_fp8_batch,
        "batched-M (<=256) fp8 weight-stream GEMM with optional split-K");
  m.def("skinny_gemm_fp8_probe", &skinny_gemm_fp8_probe,
        "fp8 tuning probe: waves, tiles");
  m.def("skinny_gemm_fp8_norm", &skinny_gemm_fp8_norm,
        "fp8-weight decode GEMM of rms-normed rows, optionally gated",
        py::arg("a"), py::arg("ss"), py::arg("parts"), py::arg("M"),
        py::arg("eps"), py::arg("qf"), py::arg("scale"), py::arg("N"),
        py::arg("K"), py::arg("glu"), py::arg("far") = false);
  m.def("skinny_gemm_fp8_block", &skinny_gemm_fp8_block,
        "waves and tiles of a block of the fp8 stream");
  m.def("skinny_gemm_fp8_parts", &skinny_gemm_fp8_parts,
        "parts of a row's sum of squares behind a residual");
  m.def("skinny_gemm_fp8_residual", &skinny_gemm_fp8_residual,
        "fp8-weight decode GEMM added to the residual stream",
        py::arg("a"), py::arg("qf"), py::arg("scale"), py::arg("N"),
        py::arg("K"), py::arg("res"), py::arg("w"), py::arg("far") = false);
  m.def("embed_rows", &embed_rows,
        "a step's first rows and their sums of squares");
  m.def("topk_cosine_host", &topk_cosine_host,
        "exact cosine top-k of host queries, normalized; result on the host");
  m.def("topk_cosine_packed", &topk_cosine_packed,
        "the same, scores and documents in one buffer");
  m.def("topk_cosine", &topk_cosine, "exact cosine top-k over the HBM index");
  m.def("hash_build", &hash_build,
        "build latest-per-key hash table from (keys, event ts)");
  m.def("hash_probe", &hash_probe,
        "probe the hash table with TTL cutoff -> row indices or -1");
  m.def("window_agg", &window_agg, "segmented (key, window) count/sum");
  m.def("anomaly_batch", &anomaly_batch, "batched AR+ridge anomaly scorer");
  register_avro(m);
  register_bpe(m);
}
