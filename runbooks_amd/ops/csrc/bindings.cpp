// Python bindings for the runbooks_amd CDNA4 (gfx950) kernel library.

#include <torch/extension.h>

at::Tensor lora_delta_(at::Tensor y, at::Tensor t, at::Tensor w, double scale, bool w_transposed);
at::Tensor lora_badd_(at::Tensor y, at::Tensor t, at::Tensor w, double scale);
at::Tensor rope_fwd(at::Tensor x, at::Tensor cos, at::Tensor sin,
                    at::Tensor positions, int64_t heads);
at::Tensor rope_bwd(at::Tensor dy, at::Tensor cos, at::Tensor sin,
                    at::Tensor positions, int64_t heads);
void adamw_step(at::Tensor p, at::Tensor g, at::Tensor m, at::Tensor v,
                double lr, double beta1, double beta2, double eps, double wd,
                int64_t step);
void adamw_step_multi(at::Tensor table, int64_t nchunks, bool p32, bool g32,
                      double lr, double beta1, double beta2, double eps,
                      double wd, int64_t step);
int64_t adamw_mt_chunk_elems();
void kv_append(at::Tensor k, at::Tensor v, at::Tensor k_cache, at::Tensor v_cache,
               at::Tensor slot_mapping);
at::Tensor paged_decode(at::Tensor q, at::Tensor k_cache, at::Tensor v_cache,
                        at::Tensor block_tables, at::Tensor seq_lens,
                        int64_t nsplit, double scale,
                        c10::optional<at::Tensor> seq_starts);
int64_t paged_decode_parts(int64_t nsplit, int64_t longest, int64_t dh,
                           int64_t group, bool transposed);
std::vector<at::Tensor> paged_decode_swz(at::Tensor q, at::Tensor k_cache,
                                         at::Tensor v_cache,
                                         at::Tensor block_tables,
                                         at::Tensor seq_lens, int64_t nsplit,
                                         double scale,
                                         c10::optional<at::Tensor> seq_starts);
std::vector<at::Tensor> flash_fwd_train_qkv(at::Tensor y, int64_t B, int64_t S,
                                            int64_t Hq, int64_t Hkv,
                                            int64_t DH, double scale);
std::vector<at::Tensor> fa_bwd_qkv(at::Tensor dout, at::Tensor y,
                                   at::Tensor out, at::Tensor lse, int64_t B,
                                   int64_t S, int64_t Hq, int64_t Hkv,
                                   int64_t DH, double scale);
void rope_qkv_(at::Tensor y, at::Tensor cos, at::Tensor sin,
               at::Tensor positions, int64_t hq, int64_t hkv, int64_t dh,
               bool inverse, c10::optional<at::Tensor> dk,
               c10::optional<at::Tensor> dv);
at::Tensor swiglu_packed_bwd(at::Tensor dh, at::Tensor y);
at::Tensor lora_down(at::Tensor x, std::vector<at::Tensor> as);
at::Tensor lora_down_columns(at::Tensor dy, std::vector<at::Tensor> bs,
                             double scale);
void lora_add_(at::Tensor y, at::Tensor t, std::vector<at::Tensor> ms,
               double scale, bool sum);
std::vector<at::Tensor> lora_grads(at::Tensor dy, at::Tensor t, at::Tensor x,
                                   at::Tensor dt, std::vector<int64_t> widths,
                                   double scale);
at::Tensor lora_grad(at::Tensor x, at::Tensor t, std::vector<int64_t> widths,
                     double scale, bool transposed);
at::Tensor flash_prefill_qkv(at::Tensor y, int64_t B, int64_t S, int64_t Hq,
                             int64_t Hkv, int64_t DH, double scale);
void qkv_rope_append_(at::Tensor y, at::Tensor cos, at::Tensor sin,
                      at::Tensor positions, at::Tensor k_cache,
                      at::Tensor v_cache, at::Tensor slot_mapping,
                      int64_t hq);
std::vector<std::vector<int64_t>> flash_walks(int64_t S, int64_t rows);
at::Tensor flash_prefill(at::Tensor q, at::Tensor k, at::Tensor v, double scale);
std::vector<at::Tensor> flash_fwd_train(at::Tensor q, at::Tensor k, at::Tensor v,
                                        double scale, bool ordered);
std::vector<at::Tensor> fa_bwd(at::Tensor dout, at::Tensor q, at::Tensor k,
                               at::Tensor v, at::Tensor out, at::Tensor lse,
                               double scale, bool ordered);
at::Tensor swiglu_fwd(at::Tensor g, at::Tensor u);
std::vector<at::Tensor> swiglu_bwd(at::Tensor dy, at::Tensor g, at::Tensor u);
std::vector<at::Tensor> cross_entropy_fwd(at::Tensor logits, at::Tensor targets,
                                          int64_t ignore_index);
at::Tensor cross_entropy_bwd(at::Tensor logits, at::Tensor targets, at::Tensor lse,
                             double gscale, int64_t ignore_index);
at::Tensor mfma_probe_32x32x16(at::Tensor a, at::Tensor b);
at::Tensor mfma_probe_16x16x32(at::Tensor a, at::Tensor b);
at::Tensor train_gemm_nt(at::Tensor a, at::Tensor b);
at::Tensor skinny_gemm(at::Tensor x, at::Tensor w);
at::Tensor skinny_gemm_fp8(at::Tensor x, at::Tensor w8, at::Tensor scale);
int64_t skinny_gemm_mmax();
at::Tensor qkv_rope_append(at::Tensor y, at::Tensor cos, at::Tensor sin,
                           at::Tensor positions, at::Tensor k_cache,
                           at::Tensor v_cache, at::Tensor slot_mapping,
                           int64_t hq);

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "runbooks_amd gfx950 HIP kernels";
  m.def("lora_delta_", &lora_delta_,
        "in-place y += scale * t[T,r<=32] @ W[N,r]^T (LoRA merge)");
  m.def("lora_badd_", &lora_badd_,
        "MFMA in-place y += scale * t[T,16] @ W[N,16]^T (LoRA B merge)");
  m.def("rope_fwd", &rope_fwd, "RoPE rotate-half forward");
  m.def("rope_bwd", &rope_bwd, "RoPE rotate-half backward (inverse rotation)");
  m.def("adamw_step", &adamw_step, "fused AdamW single-tensor step");
  m.def("adamw_step_multi", &adamw_step_multi,
        "fused AdamW multi-tensor step over a cached chunk table");
  m.def("adamw_mt_chunk_elems", &adamw_mt_chunk_elems,
        "elements per multi-tensor chunk");
  m.def("kv_append", &kv_append, "paged KV-cache append");
  m.def("paged_decode", &paged_decode, "paged GQA/MQA decode attention",
        py::arg("q"), py::arg("k_cache"), py::arg("v_cache"),
        py::arg("block_tables"), py::arg("seq_lens"), py::arg("nsplit"),
        py::arg("scale"), py::arg("seq_starts") = py::none());
  m.def("paged_decode_parts", &paged_decode_parts,
        "parts that a sequence is taken in", py::arg("nsplit"),
        py::arg("longest"), py::arg("dh"), py::arg("group"),
        py::arg("transposed"));
  m.def("paged_decode_swz", &paged_decode_swz,
        "paged decode also emitting the o_proj decode-GEMM operand",
        py::arg("q"), py::arg("k_cache"), py::arg("v_cache"),
        py::arg("block_tables"), py::arg("seq_lens"), py::arg("nsplit"),
        py::arg("scale"), py::arg("seq_starts") = py::none());
  m.def("flash_prefill", &flash_prefill, "MFMA flash-attention prefill (causal)");
  m.def("flash_walks", &flash_walks,
        "how the waves of the flash kernels walk the tiles (host only)");
  m.def("flash_fwd_train_qkv", &flash_fwd_train_qkv,
        "flash_fwd_train of q, k and v side by side in one tensor");
  m.def("fa_bwd_qkv", &fa_bwd_qkv,
        "fa_bwd of q, k and v side by side -> (dy, dk_perq, dv_perq)");
  m.def("rope_qkv_", &rope_qkv_, "RoPE of q and k within packed rows",
        py::arg("y"), py::arg("cos"), py::arg("sin"), py::arg("positions"),
        py::arg("hq"), py::arg("hkv"), py::arg("dh"),
        py::arg("inverse") = false, py::arg("dk") = py::none(),
        py::arg("dv") = py::none());
  m.def("swiglu_packed_bwd", &swiglu_packed_bwd,
        "SwiGLU backward of g and u side by side");
  m.def("lora_down", &lora_down, "t_i = x A_i^T of sibling adapters");
  m.def("lora_down_columns", &lora_down_columns, "dt_i = scale dy_i B_i");
  m.def("lora_add_", &lora_add_,
        "y_i += scale t_i B_i^T, or y += scale sum t_i A_i");
  m.def("lora_grad", &lora_grad, "scale x_i^T t_i, or scale t_i^T x");
  m.def("lora_grads", &lora_grads, "scale dy_i^T t_i, and dt_i^T x");
  m.def("flash_prefill_qkv", &flash_prefill_qkv,
        "flash_prefill of q, k and v side by side in one tensor");
  m.def("qkv_rope_append_", &qkv_rope_append_,
        "packed qkv: q and k rotated in place, k and v appended to the cache");
  m.def("flash_fwd_train", &flash_fwd_train,
        "MFMA flash-attention forward + log-sum-exp (training)", py::arg("q"),
        py::arg("k"), py::arg("v"), py::arg("scale"),
        py::arg("ordered") = false);
  m.def("fa_bwd", &fa_bwd,
        "MFMA flash-attention backward -> (dq, dk_perq, dv_perq)", py::arg("dout"),
        py::arg("q"), py::arg("k"), py::arg("v"), py::arg("out"),
        py::arg("lse"), py::arg("scale"), py::arg("ordered") = false);
  m.def("swiglu_fwd", &swiglu_fwd, "fused silu(g)*u");
  m.def("swiglu_bwd", &swiglu_bwd, "fused SwiGLU backward");
  m.def("cross_entropy_fwd", &cross_entropy_fwd, "fused CE: per-row loss + lse");
  m.def("cross_entropy_bwd", &cross_entropy_bwd, "fused CE backward -> dlogits");
  m.def("mfma_probe_16x16x32", &mfma_probe_16x16x32,
        "layout probe: one 16x16x32 bf16 MFMA as a plain matmul");
  m.def("mfma_probe_32x32x16", &mfma_probe_32x32x16,
        "layout probe: one 32x32x16 bf16 MFMA as a plain matmul");
  m.def("skinny_gemm", &skinny_gemm,
        "HBM-rate decode GEMM: y[M<=32,N] = x @ W^T (bf16)");
  m.def("skinny_gemm_mmax", &skinny_gemm_mmax);
  m.def("train_gemm_nt", &train_gemm_nt,
        "EXPERIMENTAL 256^2 8-phase bf16 GEMM (C = A @ B^T)");
  m.def("skinny_gemm_fp8", &skinny_gemm_fp8,
        "fp8-e4m3 weight-only decode GEMM with per-channel scales");
  m.def("qkv_rope_append", &qkv_rope_append,
        "packed qkv -> rope'd q + rope'd k / v appended to the paged cache");
}
