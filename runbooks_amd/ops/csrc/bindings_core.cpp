// Python bindings of the ops every served model runs (norms, gated units,
// decode GEMM, sampling).

#include <torch/extension.h>

std::vector<at::Tensor> rmsnorm_fwd(at::Tensor x, at::Tensor w, double eps);
std::vector<at::Tensor> rmsnorm_fwd_dec(at::Tensor x, at::Tensor w, double eps);
std::vector<at::Tensor> rmsnorm_res_fwd_dec(at::Tensor x, at::Tensor res, at::Tensor w, double eps);
std::vector<at::Tensor> rmsnorm_res_slab_fwd_dec(at::Tensor x, at::Tensor slabs, at::Tensor w, double eps);
std::vector<at::Tensor> rmsnorm_res32(at::Tensor x, c10::optional<at::Tensor> delta, at::Tensor w, double eps, bool want_swz, double offset);
std::vector<at::Tensor> rmsnorm_bwd(at::Tensor x, at::Tensor w, at::Tensor dy,
                                    at::Tensor inv_rms, bool need_dw,
                                    c10::optional<at::Tensor> add);
std::vector<at::Tensor> rmsnorm_res_fwd(at::Tensor x, at::Tensor res,
                                        at::Tensor w, double eps);
std::vector<at::Tensor> layernorm_res32(at::Tensor x, c10::optional<at::Tensor> delta, at::Tensor w, at::Tensor b, double eps, bool want_swz);
std::vector<at::Tensor> join_res32(at::Tensor x, c10::optional<at::Tensor> delta, at::Tensor other, bool want_swz);
at::Tensor swiglu_packed(at::Tensor y);
at::Tensor geglu_packed(at::Tensor y);
std::vector<at::Tensor> swiglu_packed_dec(at::Tensor y);
std::vector<at::Tensor> geglu_packed_dec(at::Tensor y);
at::Tensor decode_gemm_raw(at::Tensor xs, at::Tensor ws, int64_t M, int64_t N, int64_t K, bool f32, int64_t half);
at::Tensor decode_gemm(at::Tensor xs, at::Tensor ws, int64_t M, int64_t N, int64_t K, int64_t force_split, int64_t half);
at::Tensor decode_glu(at::Tensor xs, at::Tensor ws, c10::optional<at::Tensor> scale, int64_t M, int64_t N, int64_t K, bool gelu, c10::optional<at::Tensor> squares, double eps, bool rows);
at::Tensor decode_heads(at::Tensor xs, at::Tensor ws, c10::optional<at::Tensor> scale, int64_t M, int64_t N, int64_t K, c10::optional<at::Tensor> squares, double eps, at::Tensor cos, at::Tensor sin, at::Tensor positions, at::Tensor k_cache, at::Tensor v_cache, at::Tensor slots, int64_t hq);
at::Tensor decode_normed(at::Tensor xs, at::Tensor ws, c10::optional<at::Tensor> scale, int64_t M, int64_t N, int64_t K, at::Tensor squares, double eps, int64_t half);
bool rows_ends_pay(int64_t M, int64_t N, int64_t K);
bool decode_res_supported(int64_t M, int64_t N, int64_t K, bool fp8);
std::vector<at::Tensor> decode_res(at::Tensor xs, at::Tensor ws, c10::optional<at::Tensor> scale, at::Tensor res, at::Tensor norm, bool rows);
std::vector<at::Tensor> rmsnorm_res_slab_fwd(at::Tensor x, at::Tensor slabs, at::Tensor w, double eps);
at::Tensor rows_glu(at::Tensor x, at::Tensor ws, int64_t N, bool gelu, bool operand, c10::optional<at::Tensor> squares, double eps);
at::Tensor rows_heads(at::Tensor x, at::Tensor ws, int64_t N, at::Tensor cos, at::Tensor sin, at::Tensor positions, at::Tensor k_cache, at::Tensor v_cache, at::Tensor slots, int64_t hq, bool rows, c10::optional<at::Tensor> squares, double eps);
at::Tensor decode_swizzle_w(at::Tensor w, int64_t half);
at::Tensor decode_swizzle_x(at::Tensor x);
at::Tensor decode_swizzle_w8(at::Tensor w8, int64_t half);
std::vector<at::Tensor> decode_affine(at::Tensor xs, std::vector<at::Tensor> ws, std::vector<c10::optional<at::Tensor>> biases, int64_t M, int64_t act, bool operand);
bool normed_affine_supported(int64_t M, int64_t K);
bool affine_in_rows(int64_t M);
std::vector<at::Tensor> normed_affine(at::Tensor res, at::Tensor gain, at::Tensor shift, double eps, std::vector<at::Tensor> ws, std::vector<c10::optional<at::Tensor>> biases, int64_t act, bool operand, c10::optional<at::Tensor> k_cache, c10::optional<at::Tensor> v_cache, c10::optional<at::Tensor> slots);
void affine_add_(at::Tensor x, at::Tensor w, c10::optional<at::Tensor> bias, at::Tensor res);
at::Tensor embed_res32(at::Tensor tokens, at::Tensor positions, at::Tensor table, at::Tensor places);
at::Tensor sum_parts(at::Tensor parts);
bool tile_gemm_takes(at::Tensor x, at::Tensor w, bool glu);
bool tile_gemm_pays(int64_t M, int64_t N, int64_t K);
bool rows_res_supported(int64_t M, int64_t N, int64_t K);
bool parts_res_supported(int64_t N);
std::vector<at::Tensor> parts_res(at::Tensor parts, at::Tensor res, at::Tensor norm);
std::vector<at::Tensor> rows_res(at::Tensor x, at::Tensor ws, at::Tensor res, at::Tensor norm);
at::Tensor tile_lora(at::Tensor x, at::Tensor w, at::Tensor t, std::vector<at::Tensor> bs, double scale, int64_t tile);
bool tile_gemm_down_takes(at::Tensor x, at::Tensor w);
bool tile_gemm_down_pays(int64_t M, int64_t N, int64_t K);
std::vector<int64_t> tile_gemm_down_choice(int64_t M, int64_t N, int64_t K, int64_t max_parts);
at::Tensor tile_gemm_down(at::Tensor x, at::Tensor w, at::Tensor t, std::vector<at::Tensor> as, int64_t max_parts, int64_t tile, int64_t parts);
int64_t tile_gemm_parts(int64_t M, int64_t N, int64_t K);
std::vector<int64_t> tile_gemm_choice(int64_t M, int64_t N, int64_t K, int64_t max_parts);
at::Tensor tile_gemm(at::Tensor x, at::Tensor w, int64_t max_parts, int64_t glu, int64_t tile, int64_t parts);
at::Tensor decode_gemm_rows(at::Tensor x, at::Tensor ws, int64_t N, int64_t half, bool raw);
at::Tensor decode_gemm_fp8(at::Tensor xs, at::Tensor w8s, at::Tensor scale, int64_t M, int64_t N, int64_t K, bool raw, int64_t half);
int64_t decode_gemm_split(int64_t N, int64_t K);
bool decode_gemm_supported(int64_t M, int64_t N, int64_t K);
at::Tensor sample_tokens(at::Tensor logits, double temperature, int64_t seed);

// Whether tensors have been written to (their version counters), asked for
// before every replay of a captured step: 0.8 us for 129 weights, 12 in Python.
class Versions {
 public:
  explicit Versions(std::vector<at::Tensor> tensors)
      : tensors_(std::move(tensors)), sum_(sum()) {}
  bool current() const { return sum() == sum_; }

 private:
  int64_t sum() const {                 // counters only rise
    int64_t s = 0;
    for (const at::Tensor &t : tensors_) s += t._version();
    return s;
  }
  std::vector<at::Tensor> tensors_;
  int64_t sum_;
};

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  py::class_<Versions>(m, "Versions")
      .def(py::init<std::vector<at::Tensor>>())
      .def("current", &Versions::current);
  m.doc() = "runbooks_amd gfx950 HIP kernels: core serving ops";
  m.def("rmsnorm_fwd", &rmsnorm_fwd, "fused RMSNorm forward (bf16/f32)");
  m.def("rmsnorm_fwd_dec", &rmsnorm_fwd_dec,
        "RMSNorm forward + decode-GEMM operand swizzle in one pass");
  m.def("rmsnorm_res_fwd_dec", &rmsnorm_res_fwd_dec,
        "residual add + RMSNorm + decode operand swizzle in one pass");
  m.def("rmsnorm_res_slab_fwd_dec", &rmsnorm_res_slab_fwd_dec,
        "split-K slab combine + residual + RMSNorm + swizzle in one pass");
  m.def("rmsnorm_res32", &rmsnorm_res32,
        "fp32 residual += delta (or split-K slab), then RMSNorm");
  m.def("rmsnorm_bwd", &rmsnorm_bwd, "fused RMSNorm backward", py::arg("x"),
        py::arg("w"), py::arg("dy"), py::arg("inv_rms"),
        py::arg("need_dw") = true, py::arg("add") = py::none());
  m.def("rmsnorm_res_fwd", &rmsnorm_res_fwd,
        "residual sum + RMSNorm forward -> {sum, y, inv_rms}");
  m.def("layernorm_res32", &layernorm_res32,
        "fp32 residual += delta (or split-K slab), then LayerNorm");
  m.def("join_res32", &join_res32,
        "[fp32 residual + delta ; other] as a product's input");
  m.def("swiglu_packed", &swiglu_packed,
        "silu(y[:, :I]) * y[:, I:] from the fused gate/up GEMM output");
  m.def("geglu_packed", &geglu_packed,
        "packed GeGLU (tanh) epilogue [T,2I]->[T,I]");
  m.def("swiglu_packed_dec", &swiglu_packed_dec,
        "packed SwiGLU + decode-GEMM operand swizzle in one pass");
  m.def("geglu_packed_dec", &geglu_packed_dec,
        "packed GeGLU + decode-GEMM operand swizzle in one pass");
  m.def("decode_gemm_raw", &decode_gemm_raw,
        "decode GEMM returning the uncombined fp32 slab at split>1 (or always)",
        py::arg("xs"), py::arg("ws"), py::arg("M"), py::arg("N"),
        py::arg("K"), py::arg("f32") = false, py::arg("half") = 0);
  m.def("decode_gemm", &decode_gemm,
        "v2 weight-stream decode GEMM over pre-swizzled operands: "
        "y[M<=32,N] = x @ W^T (bf16), 1KiB coalesced nt weight bursts",
        py::arg("xs"), py::arg("ws"), py::arg("M"), py::arg("N"),
        py::arg("K"), py::arg("force_split") = -1, py::arg("half") = 0);
  m.def("decode_glu", &decode_glu,
        "gated unit of a decode product, as the next one's operand or rows",
        py::arg("xs"), py::arg("ws"), py::arg("scale"), py::arg("M"),
        py::arg("N"), py::arg("K"), py::arg("gelu"),
        py::arg("squares") = py::none(), py::arg("eps") = 0.0,
        py::arg("rows") = false);
  m.def("decode_heads", &decode_heads,
        "decode product of q, k and v -> rotated q, keys and values cached",
        py::arg("xs"), py::arg("ws"), py::arg("scale"), py::arg("M"),
        py::arg("N"), py::arg("K"), py::arg("squares"), py::arg("eps"),
        py::arg("cos"), py::arg("sin"), py::arg("positions"),
        py::arg("k_cache"), py::arg("v_cache"), py::arg("slots"),
        py::arg("hq"));
  m.def("decode_normed", &decode_normed,
        "decode product of an input without its norm's 1 / rms",
        py::arg("xs"), py::arg("ws"), py::arg("scale"), py::arg("M"),
        py::arg("N"), py::arg("K"), py::arg("squares"), py::arg("eps"),
        py::arg("half") = 0);
  m.def("rows_ends_pay", &rows_ends_pay);
  m.def("decode_res_supported", &decode_res_supported);
  m.def("decode_res", &decode_res,
        "residual + decode product -> {sum, normed without 1 / rms, squares}",
        py::arg("xs"), py::arg("ws"), py::arg("scale"), py::arg("res"),
        py::arg("norm"), py::arg("rows") = false);
  m.def("rmsnorm_res_slab_fwd", &rmsnorm_res_slab_fwd,
        "residual + parts of a product, then RMSNorm -> {sum, y}");
  m.def("rows_glu", &rows_glu, "decode_glu of up to 128 rows as they lie",
        py::arg("x"), py::arg("ws"), py::arg("N"), py::arg("gelu"),
        py::arg("operand") = false, py::arg("squares") = py::none(),
        py::arg("eps") = 0.0);
  m.def("rows_heads", &rows_heads,
        "decode_heads of up to 128 rows as they lie", py::arg("x"),
        py::arg("ws"), py::arg("N"), py::arg("cos"), py::arg("sin"),
        py::arg("positions"), py::arg("k_cache"), py::arg("v_cache"),
        py::arg("slots"), py::arg("hq"), py::arg("rows") = false,
        py::arg("squares") = py::none(), py::arg("eps") = 0.0);
  m.def("decode_swizzle_w", &decode_swizzle_w,
        "one-time [N,K] -> fragment-lane-major weight layout", py::arg("w"),
        py::arg("half") = 0);
  m.def("decode_swizzle_x", &decode_swizzle_x,
        "per-call x -> B-fragment lane order (zero-padded to M=32)");
  m.def("decode_swizzle_w8", &decode_swizzle_w8,
        "one-time weight layout swizzle for decode_gemm_fp8", py::arg("w8"),
        py::arg("half") = 0);
  m.def("decode_affine", &decode_affine,
        "act(x W^T + bias) to up to three matrices, or as an operand",
        py::arg("xs"), py::arg("ws"), py::arg("biases"), py::arg("M"),
        py::arg("act") = 0, py::arg("operand") = false);
  m.def("normed_affine_supported", &normed_affine_supported);
  m.def("affine_in_rows", &affine_in_rows);
  m.def("normed_affine", &normed_affine,
        "decode_affine of a residual's layer norm; k and v to the cache",
        py::arg("res"), py::arg("gain"), py::arg("shift"), py::arg("eps"),
        py::arg("ws"), py::arg("biases"), py::arg("act") = 0,
        py::arg("operand") = false, py::arg("k_cache") = py::none(),
        py::arg("v_cache") = py::none(), py::arg("slots") = py::none());
  m.def("affine_add_", &affine_add_, "residual += x W^T + bias");
  m.def("embed_res32", &embed_res32,
        "embeddings of tokens and positions, added up in fp32");
  m.def("sum_parts", &sum_parts, "fp32 [P, M, N] -> their sum [M, N] bf16");
  m.def("tile_gemm_takes", &tile_gemm_takes, py::arg("x"), py::arg("w"),
        py::arg("glu") = false, "whether tile_gemm takes x and W");
  m.def("tile_gemm_pays", &tile_gemm_pays, py::arg("M"), py::arg("N"),
        py::arg("K"), "whether it is as good as the library");
  m.def("parts_res_supported", &parts_res_supported);
  m.def("parts_res", &parts_res, "the same of fp32 parts of the product");
  m.def("rows_res_supported", &rows_res_supported);
  m.def("rows_res", &rows_res,
        "x W^T + residual of 33 to 64 rows x, times the next norm's weight, and "
        "parts of its squares");
  m.def("tile_lora", &tile_lora, py::arg("x"), py::arg("w"), py::arg("t"),
        py::arg("bs"), py::arg("scale"), py::arg("tile") = -1,
        "x @ W^T + scale t_i @ B_i^T of siblings side by side");
  m.def("tile_gemm_down_takes", &tile_gemm_down_takes, py::arg("x"),
        py::arg("w"), "whether tile_gemm_down takes x and W");
  m.def("tile_gemm_down_pays", &tile_gemm_down_pays, py::arg("M"),
        py::arg("N"), py::arg("K"), "whether it is as good as the library");
  m.def("tile_gemm_down_choice", &tile_gemm_down_choice, py::arg("M"),
        py::arg("N"), py::arg("K"), py::arg("max_parts") = 1,
        "tile, parts, tile of the rest and its first column");
  m.def("tile_gemm_down", &tile_gemm_down, py::arg("x"), py::arg("w"),
        py::arg("t"), py::arg("as_"), py::arg("max_parts") = 1,
        py::arg("tile") = -1, py::arg("parts") = 0,
        "x @ W + sum_i t_i A_i of many rows, W [K, N] (gemm_tiles.hip): bf16 "
        "[M, N], or, where max_parts > 1, possibly fp32 parts [P, M, N]");
  m.def("tile_gemm_parts", &tile_gemm_parts,
        "parts that tile_gemm makes of sums where it may");
  m.def("tile_gemm_choice", &tile_gemm_choice, py::arg("M"), py::arg("N"),
        py::arg("K"), py::arg("max_parts") = 1,
        "tile, parts, tile of the rest and its first column");
  m.def("tile_gemm", &tile_gemm, py::arg("x"), py::arg("w"),
        py::arg("max_parts") = 1, py::arg("glu") = 0, py::arg("tile") = -1,
        py::arg("parts") = 0,
        "x @ W^T of many rows (gemm_tiles.hip): bf16 [M, N], or, where max_parts "
        "allows, fp32 parts [P, M, N]; glu 1 / 2: SiLU / GELU units of [G ; U]");
  m.def("decode_gemm_rows", &decode_gemm_rows, "x [M <= 128, K] W^T",
        py::arg("x"), py::arg("ws"), py::arg("N"), py::arg("half") = 0,
        py::arg("raw") = false);
  m.def("decode_gemm_fp8", &decode_gemm_fp8,
        "decode GEMM with e4m3 weights and a scale per row",
        py::arg("xs"), py::arg("w8s"), py::arg("scale"), py::arg("M"),
        py::arg("N"), py::arg("K"), py::arg("raw") = false,
        py::arg("half") = 0);
  m.def("decode_gemm_split", &decode_gemm_split);
  m.def("decode_gemm_supported", &decode_gemm_supported);
  m.def("sample_tokens", &sample_tokens, "greedy / Gumbel-max sampling");
}
