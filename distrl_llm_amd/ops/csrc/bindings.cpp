// Python bindings for the gfx950 kernel library.
#include <torch/extension.h>
#include <vector>

torch::Tensor rmsnorm_fwd(torch::Tensor x, torch::Tensor w, double eps);
torch::Tensor rmsnorm_bwd(torch::Tensor dy, torch::Tensor x, torch::Tensor w,
                          double eps);
torch::Tensor rmsnorm_bwd_add(torch::Tensor dy, torch::Tensor x,
                              torch::Tensor w, torch::Tensor g, double eps);
std::vector<torch::Tensor> add_rmsnorm_fwd(torch::Tensor x, torch::Tensor h,
                                           torch::Tensor w, double eps);
torch::Tensor silu_mul_fwd(torch::Tensor gate, torch::Tensor up);
std::vector<torch::Tensor> silu_mul_bwd(torch::Tensor dy, torch::Tensor gate,
                                        torch::Tensor up);
void rope_inplace(torch::Tensor q, torch::Tensor k, torch::Tensor positions,
                  torch::Tensor inv_freq);
void rope_rows(torch::Tensor q, torch::Tensor k, torch::Tensor positions,
               torch::Tensor inv_freq);
void rope_scatter_qkv(torch::Tensor qkv, torch::Tensor positions,
                      torch::Tensor slots, torch::Tensor inv_freq,
                      torch::Tensor key_cache, torch::Tensor value_cache,
                      int64_t H, int64_t KV, int64_t D,
                      c10::optional<torch::Tensor> q_norm,
                      c10::optional<torch::Tensor> k_norm, double eps);
torch::Tensor silu_mul_packed(torch::Tensor gu);
torch::Tensor prefill_attention(torch::Tensor q, torch::Tensor k,
                                torch::Tensor v, torch::Tensor tile_q0,
                                torch::Tensor tile_rows, torch::Tensor tile_kv0,
                                int64_t max_len, double scale);
torch::Tensor paged_attention_decode_strided(
    torch::Tensor q, int64_t n_heads, int64_t head_dim, int64_t q_row_stride,
    torch::Tensor kcache, torch::Tensor vcache, torch::Tensor block_tables,
    torch::Tensor ctx_lens, double scale);
bool kv_copy_page(torch::Tensor key, torch::Tensor value, int64_t src, std::vector<int64_t> dst);
void kv_cache_scatter(torch::Tensor k, torch::Tensor v,
                      torch::Tensor key_cache, torch::Tensor value_cache,
                      torch::Tensor slot_mapping);
torch::Tensor paged_attention_decode(torch::Tensor q, torch::Tensor kcache,
                                     torch::Tensor vcache,
                                     torch::Tensor block_tables,
                                     torch::Tensor ctx_lens, double scale);
torch::Tensor sample_tokens(torch::Tensor logits, double temperature,
                            double top_p, int64_t top_k, torch::Tensor seeds,
                            torch::Tensor step);
std::vector<torch::Tensor> logprob_lse_fwd(torch::Tensor logits,
                                           torch::Tensor targets);
torch::Tensor logprob_loss_bwd(torch::Tensor logits, torch::Tensor targets,
                               torch::Tensor w, torch::Tensor lse,
                               c10::optional<torch::Tensor> dloss);
torch::Tensor nf4_gemm(torch::Tensor x, torch::Tensor w4f, torch::Tensor amaxf,
                       c10::optional<torch::Tensor> bias,
                       c10::optional<torch::Tensor> u,
                       c10::optional<torch::Tensor> bfrag,
                       int64_t N, int64_t K, int64_t r);
void lora_u(torch::Tensor x, torch::Tensor afrag, torch::Tensor u,
            int64_t r, int64_t ksplit);
bool skinny_gemm_takes(int64_t M, int64_t N, int64_t K);
torch::Tensor skinny_gemm(torch::Tensor x, torch::Tensor w, int64_t mode,
                          c10::optional<torch::Tensor> bias,
                          c10::optional<torch::Tensor> res,
                          c10::optional<torch::Tensor> norm_w, double eps,
                          c10::optional<torch::Tensor> u,
                          c10::optional<torch::Tensor> ub, bool tiles,
                          bool kept);
bool stream_gemm_takes(int64_t M, int64_t N, int64_t K);
torch::Tensor stream_glu(torch::Tensor x, torch::Tensor w);
torch::Tensor stream_gemm(torch::Tensor x, torch::Tensor w,
                          c10::optional<torch::Tensor> w2);
bool weights_tiles(std::vector<torch::Tensor> w, std::vector<torch::Tensor> out,
                   std::vector<int64_t> row, std::vector<bool> glu,
                   std::vector<c10::optional<torch::Tensor>> a,
                   std::vector<c10::optional<torch::Tensor>> b, std::vector<double> scale);
std::vector<torch::Tensor> add_rmsnorm_join(torch::Tensor parts,
                                            torch::Tensor res, torch::Tensor w,
                                            double eps,
                                            c10::optional<torch::Tensor> bt);
std::vector<torch::Tensor> decode_slots(torch::Tensor positions, torch::Tensor tables,
                                        int64_t block_size);
void decode_advance(torch::Tensor sampled, torch::Tensor tokens, torch::Tensor positions,
                    torch::Tensor ctx_lens, torch::Tensor limits, torch::Tensor finished,
                    torch::Tensor step, torch::Tensor out, c10::optional<int64_t> eos);
torch::Tensor paged_decode_packed(
    torch::Tensor qkv, c10::optional<torch::Tensor> bias,
    torch::Tensor positions, torch::Tensor slots, torch::Tensor inv_freq,
    torch::Tensor kcache, torch::Tensor vcache, torch::Tensor block_tables,
    torch::Tensor ctx_lens, torch::Tensor arrived, int64_t n_heads,
    double scale, c10::optional<torch::Tensor> q_norm,
    c10::optional<torch::Tensor> k_norm, double eps);
bool lora_merge(torch::Tensor w, torch::Tensor a, torch::Tensor b,
                torch::Tensor out, double scale);
bool lora_add(torch::Tensor y, torch::Tensor u, torch::Tensor m,
              double scale, c10::optional<torch::Tensor> res);
torch::Tensor mfma_probe(torch::Tensor a, torch::Tensor b);
std::vector<torch::Tensor> flash_attn_fwd(torch::Tensor q, torch::Tensor k,
                                          torch::Tensor v, double scale);
torch::Tensor flash_attention(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                              double scale);
torch::Tensor logprob_loss(torch::Tensor logits, torch::Tensor targets,
                           torch::Tensor mask, torch::Tensor rewards,
                           double scale);
torch::Tensor logprob_rows(torch::Tensor logits, torch::Tensor targets,
                           torch::Tensor w);
torch::Tensor flash_attn_varlen(torch::Tensor q, torch::Tensor k,
                                torch::Tensor v, torch::Tensor cu,
                                int64_t max_len, double scale);
std::vector<torch::Tensor> flash_varlen_fwd(torch::Tensor q, torch::Tensor k,
                                            torch::Tensor v, torch::Tensor cu,
                                            int64_t max_len, double scale,
                                            c10::optional<torch::Tensor> into);
void flash_varlen_bwd(torch::Tensor dout, torch::Tensor q, torch::Tensor k,
                      torch::Tensor v, torch::Tensor o, torch::Tensor lse,
                      torch::Tensor cu, int64_t max_len, double scale,
                      torch::Tensor dq, torch::Tensor dk, torch::Tensor dv);
std::vector<torch::Tensor> adapter_grads(std::vector<torch::Tensor> y,
                                         std::vector<torch::Tensor> p,
                                         std::vector<int64_t> by_col);
torch::Tensor product_rows(const torch::Tensor& g, const torch::Tensor& w);
bool product_py(std::vector<std::vector<torch::Tensor>> a,
                std::vector<std::vector<c10::optional<torch::Tensor>>> b,
                std::vector<c10::optional<torch::Tensor>> bias,
                std::vector<int64_t> width, std::string what,
                std::vector<torch::Tensor> out,
                c10::optional<torch::Tensor> res, int64_t tile);
torch::Tensor adapted_weight(std::vector<torch::Tensor> w,
                             std::vector<torch::Tensor> b, int64_t pad);
torch::Tensor stack_transposed(std::vector<torch::Tensor> w,
                               std::vector<int64_t> at, int64_t cols);
void rmsnorm_fwd_into(torch::Tensor x, torch::Tensor w, double eps,
                      torch::Tensor out);
void silu_mul_packed_into(torch::Tensor gu, torch::Tensor out);
void silu_mul_bwd_packed(torch::Tensor dy, torch::Tensor gu,
                         torch::Tensor dgate, torch::Tensor dup);
c10::optional<torch::Tensor> adapted_projection(
    torch::Tensor x, std::vector<torch::Tensor> W,
    std::vector<c10::optional<torch::Tensor>> bias, std::vector<torch::Tensor> A,
    std::vector<torch::Tensor> B, std::vector<double> scales,
    c10::optional<torch::Tensor> res);
c10::optional<torch::Tensor> adapted_activation(
    torch::Tensor x, std::vector<torch::Tensor> W, std::vector<torch::Tensor> A,
    std::vector<torch::Tensor> B, std::vector<double> scales);
bool silu_mul_inputs(torch::Tensor gu, torch::Tensor act, torch::Tensor m,
                     double scale, torch::Tensor out);
bool silu_mul_bwd_inputs(torch::Tensor dact, torch::Tensor gu,
                         torch::Tensor dgate, torch::Tensor dup,
                         std::vector<torch::Tensor> m,
                         std::vector<double> scales, torch::Tensor out);
bool adapter_input(torch::Tensor x, std::vector<torch::Tensor> m,
                   std::vector<double> scales, torch::Tensor out, bool k_major);
std::vector<torch::Tensor> attention_half_fwd(
    torch::Tensor x, torch::Tensor norm, double eps,
    std::vector<torch::Tensor> W, std::vector<c10::optional<torch::Tensor>> bias,
    std::vector<torch::Tensor> A, std::vector<torch::Tensor> B,
    std::vector<double> scales, c10::optional<torch::Tensor> q_norm,
    c10::optional<torch::Tensor> k_norm, double q_eps, double k_eps,
    torch::Tensor pos, torch::Tensor inv_freq, torch::Tensor cu,
    int64_t longest, double scale, int64_t head_dim);
std::vector<torch::Tensor> attention_half_bwd(
    torch::Tensor g, torch::Tensor x, torch::Tensor norm, double eps,
    std::vector<torch::Tensor> W, std::vector<torch::Tensor> A,
    std::vector<torch::Tensor> B, std::vector<double> scales,
    c10::optional<torch::Tensor> q_norm, c10::optional<torch::Tensor> k_norm,
    double q_eps, double k_eps, torch::Tensor pos, torch::Tensor back_freq,
    torch::Tensor cu, int64_t longest, double scale, torch::Tensor hu,
    torch::Tensor ou, torch::Tensor q, torch::Tensor k, torch::Tensor v,
    torch::Tensor lse, c10::optional<torch::Tensor> q0,
    c10::optional<torch::Tensor> k0, bool want_dx);
std::vector<torch::Tensor> feed_forward_half_fwd(
    torch::Tensor x, torch::Tensor norm, double eps,
    std::vector<torch::Tensor> W, std::vector<c10::optional<torch::Tensor>> bias,
    std::vector<torch::Tensor> A, std::vector<torch::Tensor> B,
    std::vector<double> scales);
std::vector<torch::Tensor> feed_forward_half_bwd(
    torch::Tensor g, torch::Tensor x, torch::Tensor norm, double eps,
    std::vector<torch::Tensor> W, std::vector<torch::Tensor> A,
    std::vector<torch::Tensor> B, std::vector<double> scales, torch::Tensor hu,
    torch::Tensor gu, torch::Tensor au, bool want_dx);
std::vector<torch::Tensor> flash_attn_bwd(torch::Tensor dout, torch::Tensor q,
                                          torch::Tensor k, torch::Tensor v,
                                          torch::Tensor o, torch::Tensor lse,
                                          double scale);
void adam8bit_step(torch::Tensor p, torch::Tensor g, torch::Tensor m_q,
                   torch::Tensor v_q, torch::Tensor m_absmax,
                   torch::Tensor v_absmax, double lr, double b1, double b2,
                   double eps, double wd, int64_t step);

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rmsnorm_fwd", &rmsnorm_fwd, "RMSNorm forward (gfx950)");
  m.def("rmsnorm_bwd", &rmsnorm_bwd, "RMSNorm backward dx (gfx950)");
  m.def("rmsnorm_bwd_add", &rmsnorm_bwd_add,
        "RMSNorm backward dx plus the residual's gradient");
  m.def("add_rmsnorm_fwd", &add_rmsnorm_fwd,
        "fused residual add + RMSNorm forward");
  m.def("silu_mul_fwd", &silu_mul_fwd, "fused SiLU*mul forward");
  m.def("silu_mul_bwd", &silu_mul_bwd, "fused SiLU*mul backward");
  m.def("rope_inplace", &rope_inplace, "fused in-place RoPE (q,k)");
  m.def("rope_rows", &rope_rows, "the same on rows of wider matrices");
  m.def("rope_scatter_qkv", &rope_scatter_qkv,
        "packed-qkv per-head norms (optional) + RoPE + paged KV scatter",
        py::arg("qkv"), py::arg("positions"), py::arg("slots"),
        py::arg("inv_freq"), py::arg("key_cache"), py::arg("value_cache"),
        py::arg("H"), py::arg("KV"), py::arg("D"),
        py::arg("q_norm") = py::none(), py::arg("k_norm") = py::none(),
        py::arg("eps") = 0.0);
  m.def("silu_mul_packed", &silu_mul_packed, "SiLU*mul on packed [gate|up]");
  m.def("paged_attention_decode_strided", &paged_attention_decode_strided,
        "paged GQA decode attention (packed-q rows)");
  m.def("prefill_attention", &prefill_attention,
        "varlen causal prefill attention (prompt phase)");
  m.def("kv_copy_page", &kv_copy_page, "copies of a page of all layers");
  m.def("kv_cache_scatter", &kv_cache_scatter, "paged KV cache scatter");
  m.def("paged_attention_decode", &paged_attention_decode,
        "paged GQA decode attention");
  m.def("sample_tokens", &sample_tokens,
        "fused temperature/top-k/top-p categorical sampling");
  m.def("logprob_lse_fwd", &logprob_lse_fwd,
        "per-token log p(target) + LSE, one streaming pass");
  m.def("logprob_loss_bwd", &logprob_loss_bwd,
        "dlogits for the masked PG/GRPO loss", py::arg("logits"),
        py::arg("targets"), py::arg("w"), py::arg("lse"),
        py::arg("dloss") = py::none());
  m.def("adam8bit_step", &adam8bit_step, "fused blockwise 8-bit Adam step");
  m.def("nf4_gemm", &nf4_gemm,
        "fused nf4-dequant MFMA GEMM with bias + LoRA-B epilogue");
  m.def("lora_u", &lora_u, "split-K LoRA A projection (u = x @ A^T)");
  m.def("skinny_gemm_takes", &skinny_gemm_takes,
        "whether skinny_gemm takes (M, N, K)");
  m.def("skinny_gemm", &skinny_gemm,
        "x W^T for few rows, with norm, bias, residual or SiLU*mul",
        py::arg("x"), py::arg("w"), py::arg("mode"),
        py::arg("bias") = py::none(), py::arg("res") = py::none(),
        py::arg("norm_w") = py::none(), py::arg("eps") = 0.0,
        py::arg("u") = py::none(), py::arg("ub") = py::none(),
        py::arg("tiles") = false, py::arg("kept") = false);
  m.def("stream_gemm_takes", &stream_gemm_takes,
        "whether stream_gemm and stream_glu take (M, N, K)");
  m.def("stream_glu", &stream_glu,
        "silu(x Wg^T) * (x Wu^T) for some tens of rows, W in tiles");
  m.def("stream_gemm", &stream_gemm,
        "fp32 partial sums of x [w; w2]^T, W in tiles", py::arg("x"),
        py::arg("w"), py::arg("w2") = py::none());
  m.def("weights_tiles", &weights_tiles, "weight_tiles of several weights, one launch for eight");
  m.def("weight_tiles",
        [](torch::Tensor w, torch::Tensor out, int64_t row, bool glu, c10::optional<torch::Tensor> a,
           c10::optional<torch::Tensor> b, double scale) {
          return weights_tiles({w}, {out}, {row}, {glu}, {a}, {b}, {scale});
        },
        "rows of W (+ scale * B A) into tiles; false: not these operands",
        py::arg("w"), py::arg("out"), py::arg("row"), py::arg("glu"),
        py::arg("a") = py::none(), py::arg("b") = py::none(),
        py::arg("scale") = 0.0);
  m.def("add_rmsnorm_join", &add_rmsnorm_join,
        "residual + partial sums (+ adapter), then RMSNorm", py::arg("parts"),
        py::arg("res"), py::arg("w"), py::arg("eps"),
        py::arg("bt") = py::none());
  m.def("adapted_projection", &adapted_projection, py::arg("x"), py::arg("w"),
        py::arg("bias"), py::arg("a"), py::arg("b"), py::arg("scales"),
        py::arg("res") = py::none(),
        "projections of one input with adapters, biases or a residual, or None");
  m.def("adapted_activation", &adapted_activation, py::arg("x"), py::arg("w"),
        py::arg("a"), py::arg("b"), py::arg("scales"),
        "SiLU*mul of two projections with adapters, or None");
  m.def("silu_mul_inputs", &silu_mul_inputs,
        "SiLU*mul with the adapter inputs of its output (tests)");
  m.def("silu_mul_bwd_inputs", &silu_mul_bwd_inputs,
        "SiLU*mul's gradients with their adapter inputs (tests)");
  m.def("adapter_input", &adapter_input, "scaled inputs of LoRA adapters");
  m.def("attention_half_fwd", &attention_half_fwd,
        "an adapted layer's attention half");
  m.def("attention_half_bwd", &attention_half_bwd);
  m.def("feed_forward_half_fwd", &feed_forward_half_fwd,
        "an adapted layer's feed-forward half");
  m.def("feed_forward_half_bwd", &feed_forward_half_bwd);
  m.def("decode_slots", &decode_slots, "cache rows and int32 positions of a step");
  m.def("decode_advance", &decode_advance, "a step's tokens into the session's state");
  m.def("paged_decode_packed", &paged_decode_packed,
        "packed [q|k|v] or its partial sums -> norms, RoPE, KV scatter, "
        "paged decode attention",
        py::arg("qkv"), py::arg("bias"), py::arg("positions"),
        py::arg("slots"), py::arg("inv_freq"), py::arg("kcache"),
        py::arg("vcache"), py::arg("block_tables"), py::arg("ctx_lens"),
        py::arg("arrived"), py::arg("n_heads"), py::arg("scale"),
        py::arg("q_norm") = py::none(), py::arg("k_norm") = py::none(),
        py::arg("eps") = 0.0);
  m.def("lora_merge", &lora_merge, "out = W + scale * B A, one pass");
  m.def("lora_add", &lora_add, "y += scale * u m (+ res) in place; false: not these operands",
        py::arg("y"), py::arg("u"), py::arg("m"), py::arg("scale"),
        py::arg("res") = c10::nullopt);
  m.def("mfma_probe", &mfma_probe, "16x16x32 bf16 MFMA mapping probe");
  m.def("flash_attn_fwd", &flash_attn_fwd,
        "causal GQA flash attention forward (returns o, lse)");
  m.def("flash_attention", &flash_attention,
        "differentiable causal GQA flash attention");
  m.def("logprob_loss", &logprob_loss, "differentiable masked PG/GRPO loss");
  m.def("logprob_rows", &logprob_rows,
        "differentiable weighted sum of token log-probabilities");
  m.def("flash_attn_varlen", &flash_attn_varlen,
        "causal GQA flash attention over a flat batch of sequences");
  m.def("flash_varlen_fwd", &flash_varlen_fwd,
        "the same with its log-sum-exp", py::arg("q"), py::arg("k"),
        py::arg("v"), py::arg("cu"), py::arg("max_len"), py::arg("scale"),
        py::arg("into") = py::none());
  m.def("flash_varlen_bwd", &flash_varlen_bwd,
        "its backward, into dq, dk and dv");
  m.def("product_rows", &product_rows, py::arg("g"), py::arg("w"),
        "g w, w (K, N) as it lies");
  m.def("product", &product_py, py::arg("a"), py::arg("b"), py::arg("bias"),
        py::arg("width"), py::arg("what"), py::arg("out"),
        py::arg("res") = py::none(), py::arg("tile") = 0,
        "sums of products with bias, residual or SiLU*mul (tests)");
  m.def("adapter_grads", &adapter_grads,
        "p^T y of several operands, summed over the rows");
  m.def("adapted_weight", &adapted_weight,
        "[W | B] of projections of one input");
  m.def("stack_transposed", &stack_transposed,
        "matrices of K columns side by side, transposed");
  m.def("rmsnorm_fwd_into", &rmsnorm_fwd_into,
        "RMSNorm forward into rows of a wider matrix");
  m.def("silu_mul_packed_into", &silu_mul_packed_into,
        "SiLU*mul of [gate | up] into rows of a wider matrix");
  m.def("silu_mul_bwd_packed", &silu_mul_bwd_packed,
        "its backward into dgate and dup");
  m.def("flash_attn_bwd", &flash_attn_bwd,
        "causal GQA flash attention backward (returns dq, dk, dv)");
}
