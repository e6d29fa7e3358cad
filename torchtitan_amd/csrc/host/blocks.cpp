// The launches of a converted linear, of the SwiGLU block and of the routed experts, forward and backward, from one
// native call each; and the single launches around them (gate, routing, log-probabilities, lists of casts), likewise.
//
// On inputs of up to a few thousand tokens these blocks wait for their host side: between two launches
// (3.3 us each) Python made operands, asked tensors for their pointers and strides and passed them on, 4 to 8 us
// a step.  Here the same entry points of the library are called with the same arguments in the same order
// (ops.py, mx_tensor.py and mx_blocks.py have them step by step); what is allocated is what is allocated there.
// Nothing is kept between calls, no pointer outlives one.  Every block's function checks that its inputs are the plain
// case -- bf16 or float32 matrices on the current GPU whose rows the casts read as they lie -- and returns None
// otherwise: the caller then takes the general path.
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <array>
#include <optional>

#include "mxfp8.h"

namespace py = pybind11;
using at::Tensor;

namespace {

// ---- the library's entry points: addresses of the symbols that the caller has loaded
struct Library {
  decltype(&mx_cast_pad) cast_pad = nullptr;
  decltype(&mx_cast_pad_many) cast_pad_many = nullptr;
  decltype(&mx_swiglu_cast_pad) swiglu = nullptr;
  decltype(&mx_swiglu_bwd_cast_pad) swiglu_bwd = nullptr;
  decltype(&mx_gemm_nt_workspace_bytes) workspace_bytes = nullptr;
  decltype(&mx_gemm_nt_ld) gemm = nullptr;
  decltype(&mx_gemm_nt_f32_ld) gemm_f32 = nullptr;
  decltype(&mx_gemm_nt_shared_a_ld) shared_a = nullptr;
  decltype(&mx_gemm_nt_shared_b_ld) shared_b = nullptr;
  decltype(&mx_gemm_nt_pair_ld) pair = nullptr;
  decltype(&mx_gemm_nt_pair_workspace_bytes) pair_workspace_bytes = nullptr;
  decltype(&mx_gemm_nt_pair_ws) pair_split = nullptr;
  decltype(&mx_few_rows) few_rows = nullptr;
  decltype(&mx_route_fill) route_fill = nullptr;
  decltype(&mx_cast_rows_gathered) rows_gathered = nullptr;
  decltype(&mx_swiglu_cast_dim0_dim1_ld) swiglu_dense = nullptr;
  decltype(&mx_swiglu_bwd_cast_dim0_dim1_ld) swiglu_bwd_dense = nullptr;
  decltype(&mx_grouped_gemm_2d3d) grouped = nullptr;
  decltype(&mx_grouped_gemm_2d3d_shared_a) grouped_shared_a = nullptr;
  decltype(&mx_grouped_gemm_2d3d_pair) grouped_pair = nullptr;
  decltype(&mx_grouped_gemm_2d2d) grouped_wgrad = nullptr;
  decltype(&mx_grouped_gemm_2d2d_shared_b) grouped_wgrad_two = nullptr;
  decltype(&mx_moe_combine) combine = nullptr;
  decltype(&mx_moe_combine_dot) combine_dot = nullptr;
  decltype(&mx_gate_logits) gate_logits = nullptr;
  decltype(&mx_gate_dx) gate_dx = nullptr;
  decltype(&mx_gate_dw_workspace) gate_dw_workspace = nullptr;
  decltype(&mx_gate_dw) gate_dw = nullptr;
  decltype(&mx_route_topk) route_topk = nullptr;
  decltype(&mx_route_topk_bwd) route_topk_bwd = nullptr;
  decltype(&mx_token_logprob_fwd_split) logprob_fwd = nullptr;
  decltype(&mx_token_logprob_bwd_any) logprob_bwd = nullptr;
  decltype(&mx_cast_rows_many) rows_many = nullptr;
  decltype(&mx_dequant_many) dequant_many = nullptr;
} lib;
PyObject* check_status = nullptr;  // _lib.check, never released

void bind(const py::dict& addresses, const py::object& check) {
  auto set = [&](const char* name, auto& fn) {
    fn = reinterpret_cast<std::decay_t<decltype(fn)>>(addresses[name].cast<uintptr_t>());
  };
  set("mx_cast_pad", lib.cast_pad);
  set("mx_cast_pad_many", lib.cast_pad_many);
  set("mx_swiglu_cast_pad", lib.swiglu);
  set("mx_swiglu_bwd_cast_pad", lib.swiglu_bwd);
  set("mx_gemm_nt_workspace_bytes", lib.workspace_bytes);
  set("mx_gemm_nt_ld", lib.gemm);
  set("mx_gemm_nt_f32_ld", lib.gemm_f32);
  set("mx_gemm_nt_shared_a_ld", lib.shared_a);
  set("mx_gemm_nt_shared_b_ld", lib.shared_b);
  set("mx_gemm_nt_pair_ld", lib.pair);
  set("mx_gemm_nt_pair_workspace_bytes", lib.pair_workspace_bytes);
  set("mx_gemm_nt_pair_ws", lib.pair_split);
  set("mx_few_rows", lib.few_rows);
  set("mx_route_fill", lib.route_fill);
  set("mx_cast_rows_gathered", lib.rows_gathered);
  set("mx_swiglu_cast_dim0_dim1_ld", lib.swiglu_dense);
  set("mx_swiglu_bwd_cast_dim0_dim1_ld", lib.swiglu_bwd_dense);
  set("mx_grouped_gemm_2d3d", lib.grouped);
  set("mx_grouped_gemm_2d3d_shared_a", lib.grouped_shared_a);
  set("mx_grouped_gemm_2d3d_pair", lib.grouped_pair);
  set("mx_grouped_gemm_2d2d", lib.grouped_wgrad);
  set("mx_grouped_gemm_2d2d_shared_b", lib.grouped_wgrad_two);
  set("mx_moe_combine", lib.combine);
  set("mx_moe_combine_dot", lib.combine_dot);
  set("mx_gate_logits", lib.gate_logits);
  set("mx_gate_dx", lib.gate_dx);
  set("mx_gate_dw_workspace", lib.gate_dw_workspace);
  set("mx_gate_dw", lib.gate_dw);
  set("mx_route_topk", lib.route_topk);
  set("mx_route_topk_bwd", lib.route_topk_bwd);
  set("mx_token_logprob_fwd_split", lib.logprob_fwd);
  set("mx_token_logprob_bwd_any", lib.logprob_bwd);
  set("mx_cast_rows_many", lib.rows_many);
  set("mx_dequant_many", lib.dequant_many);
  check_status = check.ptr();
  Py_INCREF(check_status);
}

// Python's other threads run while a call allocates and launches, as they do under ctypes: a launch waits where the
// queue is full.  Reset before Python objects are made.
using Unlocked = std::optional<py::gil_scoped_release>;

void checked(int status, const char* name) {
  if (!status) return;
  py::gil_scoped_acquire locked;
  py::reinterpret_borrow<py::object>(check_status)(status, name);  // raises
}

// What a block needs until it returns.  Small blocks, whose host side decides, take all of it from one allocation
// (1.2 us each; routed experts backward: ten); larger ones as they did, piece by piece, so that the allocator's blocks
// keep their sizes.
class Scratch {
 public:
  Scratch(int64_t total, const Tensor& like) : bytes_(like.options().dtype(at::kByte)) {
    if (total <= kTogether) all_ = at::empty({total}, bytes_);
  }
  uint8_t* take(int64_t bytes) {
    bytes = padded(bytes);
    if (all_.defined()) {
      TORCH_INTERNAL_ASSERT(used_ + bytes <= all_.numel());
      uint8_t* const p = all_.data_ptr<uint8_t>() + used_;
      used_ += bytes;
      return p;
    }
    pieces_.push_back(at::empty({bytes}, bytes_));
    return pieces_.back().data_ptr<uint8_t>();
  }
  static int64_t padded(int64_t bytes) { return (bytes + 511) & ~int64_t{511}; }

 private:
  static constexpr int64_t kTogether = int64_t{64} << 20;
  at::TensorOptions bytes_;
  Tensor all_;
  int64_t used_ = 0;
  std::vector<Tensor> pieces_;
};

// ---- operands (ops.Operand): codes [rows, cols up to 128], rows `ld` bytes apart, then the scales
struct Operand {
  Tensor buf;
  int64_t rows, k, ld, at, scales_at, depth;
  uint8_t* codes() const { return buf.data_ptr<uint8_t>() + at; }
  uint8_t* scales() const { return buf.data_ptr<uint8_t>() + scales_at; }
  py::tuple layout() const { return py::make_tuple(rows, k, ld, at, scales_at, depth); }
};

int64_t up128(int64_t n) { return (n + 127) & ~int64_t{127}; }

Operand layout_of(int64_t rows, int64_t cols, int64_t pad) {
  const int64_t k = up128(cols), ld = k + pad;
  return {Tensor(), rows, k, ld, 0, (rows * ld + 255) & ~int64_t{255}, cols};
}
Operand make(int64_t rows, int64_t cols, int64_t pad, const Tensor& like) {
  Operand o = layout_of(rows, cols, pad);
  o.buf = at::empty({o.scales_at + up128(rows) * (o.k / 32)}, like.options().dtype(at::kByte));
  return o;
}
std::array<Operand, 2> make_pair(int64_t rows, int64_t cols, int64_t pad, const Tensor& like) {
  Operand a = layout_of(rows, cols, pad), b = a;
  const int64_t scales = up128(rows) * (a.k / 32);
  a.scales_at = (2 * rows * a.ld + 255) & ~int64_t{255};
  b.at = rows * a.ld;
  b.scales_at = a.scales_at + scales;
  a.buf = b.buf = at::empty({a.scales_at + 2 * scales}, like.options().dtype(at::kByte));
  return {a, b};
}

// N operands of rows x cols, in one buffer where they are small (see Scratch)
template <size_t N>
std::array<Operand, N> make_all(const std::array<std::array<int64_t, 2>, N>& sides, int64_t pad, const Tensor& like) {
  std::array<Operand, N> all;
  int64_t total = 0;
  for (size_t i = 0; i < N; ++i) {
    Operand& o = all[i] = layout_of(sides[i][0], sides[i][1], pad);
    const int64_t bytes = o.scales_at + up128(o.rows) * (o.k / 32);
    o.at += total;
    o.scales_at += total;
    total += Scratch::padded(bytes);
  }
  if (total > (int64_t{64} << 20)) {
    for (size_t i = 0; i < N; ++i) all[i] = make(sides[i][0], sides[i][1], pad, like);
    return all;
  }
  const Tensor buf = at::empty({total}, like.options().dtype(at::kByte));
  for (Operand& o : all) o.buf = buf;
  return all;
}

// A saved operand of `rows` rows and a contraction of `cols`, from the buffer that a backward gets back (hooks on
// saved tensors may have made it anew) and the layout that the forward kept: false unless it is what the products
// of this call take, on the GPU of `like`.  (ops.saved_operand has the general case.)
using Layout = std::array<int64_t, 6>;
bool saved_operand(Operand& o, const Tensor& buf, const Layout& layout, int64_t rows, int64_t cols, int64_t pad, const Tensor& like) {
  const auto [r, k, ld, at, scales_at, depth] = layout;
  o = {buf, r, k, ld, at, scales_at, depth};
  return r == rows && depth == cols && k == up128(cols) && ld == k + pad && buf.scalar_type() == at::kByte &&
         buf.device() == like.device() && buf.is_contiguous() && buf.numel() >= scales_at + up128(rows) * (k / 32);
}

// A matrix that the casts read as it lies (ops._operand_input returns it unchanged)
bool plain(const Tensor& t) {
  if (!t.is_cuda() || t.dim() != 2) return false;
  const auto type = t.scalar_type();
  if (type != at::kBFloat16 && type != at::kFloat) return false;
  const int64_t size = type == at::kFloat ? 4 : 2;
  return t.size(0) > 0 && t.size(1) > 0 && t.size(1) % 32 == 0 && t.stride(1) == 1 && t.stride(0) >= t.size(1) &&
         t.stride(0) * size % 16 == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}
bool plain_weight(const Tensor& w, const Tensor& x) {
  return plain(w) && w.is_contiguous() && w.device() == x.device();
}
bool on_current_device(const Tensor& t) { return t.device().index() == c10::hip::current_device(); }
hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void add_cast(std::array<int64_t, 8 * MX_CAST_PAD_MANY_FIELDS>& table, int64_t& n, const Tensor& x, const Operand& r,
              const Operand& c) {
  const int64_t entry[MX_CAST_PAD_MANY_FIELDS] = {
      reinterpret_cast<int64_t>(x.data_ptr()), x.scalar_type() == at::kFloat, 1, x.size(0), x.size(1), x.stride(0),
      reinterpret_cast<int64_t>(r.codes()), r.ld, reinterpret_cast<int64_t>(r.scales()),
      reinterpret_cast<int64_t>(c.codes()), c.ld, reinterpret_cast<int64_t>(c.scales())};
  std::copy(entry, entry + MX_CAST_PAD_MANY_FIELDS, table.begin() + MX_CAST_PAD_MANY_FIELDS * n++);
}

// ops._gemm_operands, into rows of `out` (2-D, unit inner stride)
void gemm_into(const Operand& a, const Operand& b, const Tensor& out, hipStream_t st) {
  const int64_t need = lib.workspace_bytes(a.rows, b.rows, a.k);
  const Tensor ws = need ? at::empty({need}, a.buf.options()) : Tensor();
  checked(lib.gemm(a.codes(), a.scales(), b.codes(), b.scales(), out.data_ptr(), a.rows, b.rows, a.k, a.ld, out.stride(0),
                   need ? ws.data_ptr() : nullptr, need, st),
          "mx_gemm_nt_ld");
}
// ops.mx_gemm_nt_as
Tensor gemm(const Operand& a, const Operand& b, const Tensor& like, hipStream_t st, at::ScalarType type = at::kBFloat16) {
  const int64_t M = a.rows, N = b.rows;
  if (type == at::kFloat && M > 64 && N > 128 && N % 8 == 0 && std::max(N * 1024, a.ld * 256) < (int64_t{1} << 31)) {
    Tensor out = at::empty({M, N}, like.options().dtype(at::kFloat));
    const int64_t need = lib.workspace_bytes(M, N, a.k);
    const Tensor ws = need ? at::empty({need}, a.buf.options()) : Tensor();
    checked(lib.gemm_f32(a.codes(), a.scales(), b.codes(), b.scales(), out.data_ptr<float>(), M, N, a.k, a.ld, N,
                         need ? ws.data_ptr() : nullptr, need, st),
            "mx_gemm_nt_f32_ld");
    return out;
  }
  Tensor out = at::empty({M, N}, like.options().dtype(at::kBFloat16));
  gemm_into(a, b, out, st);
  return type == at::kBFloat16 ? out : out.to(type);
}

bool persistent_shape(int64_t M, int64_t N) { return M > 128 && N > 128 && N % 8 == 0; }

// ---- the linear ----------------------------------------------------------------------------------
// (y, row-wise x, column-wise x, column-wise W) of y = x W^T; operands as (buffer, layout)
py::object linear_forward(const Tensor& x, const Tensor& w, int mode, int64_t pad) {
  if (!plain(x) || !plain_weight(w, x) || x.size(1) != w.size(1) || !on_current_device(x)) return py::none();
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  hipStream_t st = stream_of(x);
  Unlocked unlocked(std::in_place);
  const Operand xr = make(M, K, pad, x), xc = make(K, M, pad, x), wr = make(N, K, pad, x), wc = make(K, N, pad, x);
  std::array<int64_t, 8 * MX_CAST_PAD_MANY_FIELDS> table;
  int64_t n = 0;
  add_cast(table, n, x, xr, xc);
  add_cast(table, n, w, wr, wc);
  checked(lib.cast_pad_many(n, table.data(), mode, st), "mx_cast_pad_many");
  const Tensor y = gemm(xr, wr, x, st);
  unlocked.reset();
  return py::make_tuple(y, xr.buf, xr.layout(), xc.buf, xc.layout(), wc.buf, wc.layout());
}

// (dx, dW) from dy and linear_forward's column-wise operands
py::object linear_backward(const Tensor& dy, const Tensor& x_buf, const Layout& x_layout, const Tensor& w_buf,
                           const Layout& w_layout, int mode, int64_t pad, bool dx_f32, bool dw_f32) {
  if (!plain(dy) || !on_current_device(dy)) return py::none();
  const int64_t M = dy.size(0), N = dy.size(1), K = x_layout[0];
  Operand x, w;
  if (!saved_operand(x, x_buf, x_layout, K, M, pad, dy) || !saved_operand(w, w_buf, w_layout, K, N, pad, dy)) return py::none();
  hipStream_t st = stream_of(dy);
  Unlocked unlocked(std::in_place);
  const auto [r, c] = make_all<2>({{{M, N}, {N, M}}}, pad, dy);
  checked(lib.cast_pad(dy.data_ptr(), dy.scalar_type() == at::kFloat, M, N, dy.stride(0), r.codes(), r.ld, r.scales(),
                       c.codes(), c.ld, c.scales(), mode, st),
          "mx_cast_pad");
  const Tensor dx = gemm(r, w, dy, st, dx_f32 ? at::kFloat : at::kBFloat16);
  const Tensor dw = gemm(c, x, dy, st, dw_f32 ? at::kFloat : at::kBFloat16);
  unlocked.reset();
  return py::make_tuple(dx, dw);
}

// y = x W^T without gradients, W's row-wise operand given (its buffers and layout): (y, row-wise x or None).
// `few`: by the product that casts x itself (ops.few_rows_ok).
py::object linear_apply(const Tensor& x, const Tensor& w_buf, const Tensor& w_scales, const Layout& layout,
                        int mode, bool few) {
  const auto [N, k, ld, at, scales_at, depth] = layout;
  if (!plain(x) || x.size(1) != depth || ld % 128 || w_buf.device() != x.device() || !on_current_device(x)) return py::none();
  const int64_t M = x.size(0), K = x.size(1);
  hipStream_t st = stream_of(x);
  Unlocked unlocked(std::in_place);
  const uint8_t* codes = w_buf.data_ptr<uint8_t>() + at;
  const uint8_t* scales = w_scales.data_ptr<uint8_t>() + scales_at;
  if (few) {
    const Tensor y = at::empty({M, N}, x.options());
    checked(lib.few_rows(x.data_ptr(), M, K, x.stride(0), codes, scales, nullptr, nullptr, N, ld, y.data_ptr(), nullptr, N,
                         mode, st),
            "mx_few_rows");
    unlocked.reset();
    return py::make_tuple(y, py::none(), py::none());
  }
  const Operand xr = make(M, K, ld - k, x);
  checked(lib.cast_pad(x.data_ptr(), x.scalar_type() == at::kFloat, M, K, x.stride(0), xr.codes(), xr.ld, xr.scales(), nullptr,
                       0, nullptr, mode, st),
          "mx_cast_pad");
  const Tensor y = at::empty({M, N}, x.options().dtype(at::kBFloat16));
  const int64_t need = lib.workspace_bytes(M, N, k);
  const Tensor ws = need ? at::empty({need}, xr.buf.options()) : Tensor();
  checked(lib.gemm(xr.codes(), xr.scales(), codes, scales, y.data_ptr(), M, N, k, ld, N, need ? ws.data_ptr() : nullptr, need,
                   st),
          "mx_gemm_nt_ld");
  unlocked.reset();
  return py::make_tuple(y, xr.buf, xr.layout());
}

// ---- the SwiGLU block ----------------------------------------------------------------------------
// (y, h13, then row-wise x and column-wise W2, x, g, W1, W3 as (buffer, layout)) of
// y = (silu(x W1^T) * (x W3^T)) W2^T
py::object ffn_forward(const Tensor& x, const Tensor& w1, const Tensor& w3, const Tensor& w2, int mode, int64_t pad) {
  if (!plain(x) || x.scalar_type() != at::kBFloat16 || !plain_weight(w1, x) || !plain_weight(w3, x) ||
      !plain_weight(w2, x) || !on_current_device(x))
    return py::none();
  const int64_t M = x.size(0), D = x.size(1), H = w1.size(0), O = w2.size(0);
  if (w1.size(1) != D || w3.size(1) != D || w3.size(0) != H || w2.size(1) != H) return py::none();
  hipStream_t st = stream_of(x);
  Unlocked unlocked(std::in_place);
  const Operand xr = make(M, D, pad, x), xc = make(D, M, pad, x);
  const Operand w1c = make(D, H, pad, x), w3c = make(D, H, pad, x), w2c = make(H, O, pad, x);
  const auto [w1r, w3r, w2r, gr] = make_all<4>({{{H, D}, {H, D}, {O, H}, {M, H}}}, pad, x);
  std::array<int64_t, 8 * MX_CAST_PAD_MANY_FIELDS> table;
  int64_t n = 0;
  add_cast(table, n, x, xr, xc);
  add_cast(table, n, w1, w1r, w1c);
  add_cast(table, n, w3, w3r, w3c);
  add_cast(table, n, w2, w2r, w2c);
  checked(lib.cast_pad_many(n, table.data(), mode, st), "mx_cast_pad_many");
  const Tensor h13 = at::empty({2, M, H}, x.options());
  char* const h1 = static_cast<char*>(h13.data_ptr());
  char* const h3 = h1 + 2 * M * H;
  if (persistent_shape(M, H)) {
    checked(lib.shared_a(xr.codes(), xr.scales(), w1r.codes(), w1r.scales(), w3r.codes(), w3r.scales(), h1, h3, M, H, xr.k,
                         xr.ld, H, st),
            "mx_gemm_nt_shared_a_ld");
  } else {
    gemm_into(xr, w1r, h13[0], st);
    gemm_into(xr, w3r, h13[1], st);
  }
  const Operand gc = make(H, M, pad, x);
  checked(lib.swiglu(h1, h3, M, H, H, H, gr.codes(), gr.ld, gr.scales(), gc.codes(), gc.ld, gc.scales(), mode, st),
          "mx_swiglu_cast_pad");
  const Tensor y = gemm(gr, w2r, x, st);
  unlocked.reset();
  return py::make_tuple(y, h13, xr.buf, xr.layout(), w2c.buf, w2c.layout(), xc.buf, xc.layout(), gc.buf, gc.layout(),
                        w1c.buf, w1c.layout(), w3c.buf, w3c.layout());
}

// (dx, dW1, dW2, dW3), bf16, from dy and what ffn_forward returned: h13 and the column-wise W2, x, g, W1, W3
py::object ffn_backward(const Tensor& dy, const Tensor& h13, const std::array<Tensor, 5>& bufs,
                        const std::array<Layout, 5>& layouts, int64_t D, int mode, int64_t pad) {
  if (!plain(dy) || !on_current_device(dy) || h13.dim() != 3 || !h13.is_contiguous() || h13.scalar_type() != at::kBFloat16 ||
      h13.device() != dy.device() || h13.size(0) != 2 || h13.size(1) != dy.size(0))
    return py::none();
  const int64_t M = dy.size(0), O = dy.size(1), H = h13.size(2);
  const std::array<std::array<int64_t, 2>, 5> sides{{{H, O}, {D, M}, {H, M}, {D, H}, {D, H}}};
  std::array<Operand, 5> saved;
  for (int i = 0; i < 5; ++i)
    if (!saved_operand(saved[i], bufs[i], layouts[i], sides[i][0], sides[i][1], pad, dy)) return py::none();
  const auto& [w2, x, g, w1, w3] = saved;
  hipStream_t st = stream_of(dy);
  Unlocked unlocked(std::in_place);
  const auto [r, c] = make_all<2>({{{M, O}, {O, M}}}, pad, dy);
  checked(lib.cast_pad(dy.data_ptr(), dy.scalar_type() == at::kFloat, M, O, dy.stride(0), r.codes(), r.ld, r.scales(),
                       c.codes(), c.ld, c.scales(), mode, st),
          "mx_cast_pad");
  const Tensor dg = gemm(r, w2, dy, st);
  const auto [ra, rb] = make_pair(M, H, pad, dy);
  const auto [ca, cb] = make_pair(H, M, pad, dy);
  const char* h1 = static_cast<const char*>(h13.data_ptr());
  checked(lib.swiglu_bwd(dg.data_ptr(), h1, h1 + 2 * M * H, M, H, H, H, H, ra.codes(), ra.ld, ra.scales(), ca.codes(),
                         ca.ld, ca.scales(), mode, st),
          "mx_swiglu_bwd_cast_pad");
  const Tensor dw13 = at::empty({2, H, D}, h13.options());
  if (persistent_shape(H, D)) {
    char* out = static_cast<char*>(dw13.data_ptr());
    checked(lib.shared_b(ca.codes(), ca.scales(), cb.codes(), cb.scales(), x.codes(), x.scales(), out, out + 2 * H * D, H, D,
                         x.k, x.ld, D, st),
            "mx_gemm_nt_shared_b_ld");
  } else {
    gemm_into(ca, x, dw13[0], st);
    gemm_into(cb, x, dw13[1], st);
  }
  const Tensor dw2 = gemm(c, g, dy, st);
  Tensor dx;
  if (persistent_shape(M, D)) {
    dx = at::empty({M, D}, h13.options());
    if (const int64_t need = lib.pair_workspace_bytes(M, D, ra.k)) {
      const Tensor ws = at::empty({need}, ra.buf.options());
      checked(lib.pair_split(ra.codes(), ra.scales(), w1.codes(), w1.scales(), rb.codes(), rb.scales(), w3.codes(),
                             w3.scales(), dx.data_ptr(), M, D, ra.k, ra.ld, D, ws.data_ptr(), need, st),
              "mx_gemm_nt_pair_ws");
    } else {
      checked(lib.pair(ra.codes(), ra.scales(), w1.codes(), w1.scales(), rb.codes(), rb.scales(), w3.codes(), w3.scales(),
                       dx.data_ptr(), M, D, ra.k, ra.ld, D, st),
              "mx_gemm_nt_pair_ld");
    }
  } else {
    dx = gemm(ra, w1, dy, st) + gemm(rb, w3, dy, st);
  }
  unlocked.reset();
  return py::make_tuple(dx, dw13.select(0, 0), dw2, dw13.select(0, 1));
}

// ---- the routed experts --------------------------------------------------------------------------
// Dense codes [rows, cols] (or a stack of them) and their scales in MFMA order, rows and cols whole 128s but for
// `rows` of an activation (ops.MXData).
struct Codes {
  Tensor codes, scales;
  const uint8_t* c() const { return codes.data_ptr<uint8_t>(); }
  const uint8_t* s() const { return scales.data_ptr<uint8_t>(); }
  uint8_t* c() { return codes.data_ptr<uint8_t>(); }
  uint8_t* s() { return scales.data_ptr<uint8_t>(); }
};
Codes make_codes(int64_t rows, int64_t cols, const Tensor& like) {
  const auto bytes = like.options().dtype(at::kByte);
  return {at::empty({rows, cols}, bytes), at::empty({up128(rows) * ((cols / 32 + 1) / 2 * 2)}, bytes)};
}
Codes make_stack(int64_t G, int64_t rows, int64_t cols, const Tensor& like) {
  const auto bytes = like.options().dtype(at::kByte);
  return {at::empty({G, rows, cols}, bytes), at::empty({G * rows * (cols / 32)}, bytes)};
}
// ... of a Scratch
struct Lent {
  uint8_t *c, *s;
};
void add_stack(std::array<int64_t, 8 * MX_CAST_PAD_MANY_FIELDS>& table, int64_t& n, const Tensor& w, const Lent& r, Codes& c) {
  const int64_t entry[MX_CAST_PAD_MANY_FIELDS] = {
      reinterpret_cast<int64_t>(w.data_ptr()), w.scalar_type() == at::kFloat, w.size(0), w.size(1), w.size(2), w.size(2),
      reinterpret_cast<int64_t>(r.c), w.size(2), reinterpret_cast<int64_t>(r.s),
      reinterpret_cast<int64_t>(c.c()), w.size(1), reinterpret_cast<int64_t>(c.s())};
  std::copy(entry, entry + MX_CAST_PAD_MANY_FIELDS, table.begin() + MX_CAST_PAD_MANY_FIELDS * n++);
}
bool plain_stack(const Tensor& w, int64_t G, int64_t rows, int64_t cols, const Tensor& x) {
  return w.dim() == 3 && w.size(0) == G && w.size(1) == rows && w.size(2) == cols && w.is_contiguous() &&
         (w.scalar_type() == at::kBFloat16 || w.scalar_type() == at::kFloat) && w.device() == x.device() &&
         reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0;
}
bool plain_list(const Tensor& t, at::ScalarType type, const Tensor& x) {
  return t.scalar_type() == type && t.is_contiguous() && t.device() == x.device();
}

// (out, the slots of mx_blocks.ROUTED_SAVED) on x [T, D] for all gradients, from the router's choices; hidden and
// model size whole 128s.
py::object routed_forward(const Tensor& x, const Tensor& scores, const Tensor& w1, const Tensor& w3, const Tensor& w2,
                          const Tensor& selected, const Tensor& block_counts, const Tensor& counts, int64_t alignment,
                          int64_t multiple, int mode, bool score_before) {
  if (!plain(x) || x.scalar_type() != at::kBFloat16 || !on_current_device(x) || w1.dim() != 3) return py::none();
  const int64_t T = x.size(0), D = x.size(1), G = w1.size(0), H = w1.size(1);
  if (D % 128 || H % 128 || !plain_stack(w1, G, H, D, x) || !plain_stack(w3, G, H, D, x) || !plain_stack(w2, G, D, H, x) ||
      scores.dim() != 2 || scores.size(0) != T || !plain_list(scores, at::kFloat, x) || !plain_list(selected, at::kLong, x) ||
      selected.sizes() != scores.sizes() || !plain_list(block_counts, at::kInt, x) || !plain_list(counts, at::kLong, x) ||
      counts.numel() != G || block_counts.numel() < (T + 15) / 16 * G || alignment % 32 || multiple % 128 || multiple % alignment)
    return py::none();
  const int64_t k = scores.size(1);
  int64_t R = (T * k + alignment * G + multiple - 1) / multiple * multiple;  // ops.plan_length
  if (multiple == 128 && R % 512 == 0 && ((R & (R - 1)) != 0 || R >= 65536)) R += multiple;
  hipStream_t st = stream_of(x);
  Unlocked unlocked(std::in_place);
  const Tensor offs = at::empty({G}, x.options().dtype(at::kInt)), src_row = at::empty({R}, x.options().dtype(at::kLong)),
               row_score = at::empty({R}, x.options().dtype(at::kFloat)),
               pos = at::empty({T, k}, x.options().dtype(at::kLong));
  const int32_t* ends = offs.data_ptr<int32_t>();
  checked(lib.route_fill(selected.data_ptr<int64_t>(), scores.data_ptr<float>(), T, k, G, block_counts.data_ptr<int32_t>(),
                         counts.data_ptr<int64_t>(), R, alignment, offs.data_ptr<int32_t>(), src_row.data_ptr<int64_t>(),
                         row_score.data_ptr<float>(), pos.data_ptr<int64_t>(), st),
          "mx_route_fill");
  const auto scale_bytes = [](int64_t rows, int64_t cols) { return up128(rows) * (cols / 32); };
  const int64_t weight = G * D * H, weight_s = weight / 32, xr_s = scale_bytes(R, D), gr_s = scale_bytes(R, H);
  Scratch scratch(Scratch::padded(R * D) + Scratch::padded(xr_s) + 3 * (Scratch::padded(weight) + Scratch::padded(weight_s)) +
                      Scratch::padded(R * H) + Scratch::padded(gr_s),
                  x);
  const auto taken = [&](int64_t codes, int64_t scales) { return Lent{scratch.take(codes), scratch.take(scales)}; };
  const Lent xr = taken(R * D, xr_s);
  Codes xc = make_codes(D, R, x);
  checked(lib.rows_gathered(x.data_ptr(), src_row.data_ptr<int64_t>(), score_before ? row_score.data_ptr<float>() : nullptr, T,
                            R, D, x.stride(0), xr.c, xr.s, xc.c(), xc.s(), mode, MX_SCALES_MFMA, st),
          "mx_cast_rows_gathered");
  const Lent w1r = taken(weight, weight_s), w3r = taken(weight, weight_s), w2r = taken(weight, weight_s);
  Codes w1c = make_stack(G, D, H, x), w3c = make_stack(G, D, H, x), w2c = make_stack(G, H, D, x);
  std::array<int64_t, 8 * MX_CAST_PAD_MANY_FIELDS> table;
  int64_t n = 0;
  add_stack(table, n, w1, w1r, w1c);
  add_stack(table, n, w3, w3r, w3c);
  add_stack(table, n, w2, w2r, w2c);
  checked(lib.cast_pad_many(n, table.data(), mode, st), "mx_cast_pad_many");
  const Tensor h13 = at::empty({2, R, H}, x.options());
  char* const h1 = static_cast<char*>(h13.data_ptr());
  char* const h3 = h1 + 2 * R * H;
  checked(lib.grouped_shared_a(xr.c, xr.s, w1r.c, w1r.s, w3r.c, w3r.s, ends, h1, h3, R, H, D, G, H, st),
          "mx_grouped_gemm_2d3d_shared_a");
  const Lent gr = taken(R * H, gr_s);
  Codes gc = make_codes(H, R, x);
  checked(lib.swiglu_dense(h1, h3, R, H, H, H, gr.c, H, gr.s, gc.c(), R, gc.s(), nullptr, mode, MX_SCALES_MFMA, st),
          "mx_swiglu_cast_dim0_dim1_ld");
  const Tensor yp = at::empty({R, D}, x.options()), out = at::empty({T, D}, x.options());
  checked(lib.grouped(gr.c, gr.s, w2r.c, w2r.s, ends, yp.data_ptr(), R, D, H, G, D, MX_SCALES_MFMA, st),
          "mx_grouped_gemm_2d3d");
  checked(lib.combine(yp.data_ptr(), nullptr, R, D, pos.data_ptr<int64_t>(), score_before ? nullptr : scores.data_ptr<float>(),
                      T, k, D, out.data_ptr(), D, st),
          "mx_moe_combine");
  unlocked.reset();
  return py::make_tuple(out, py::make_tuple(offs, src_row, row_score, pos, scores, h13, w2c.codes, w2c.scales, xc.codes,
                                            xc.scales, gc.codes, gc.scales, w1c.codes, w1c.scales, w3c.codes, w3c.scales,
                                            score_before ? x : yp));
}

// (dx, d scores, dW1, dW2, dW3) from dout [T, D] and those slots; at most 16 choices a token
py::object routed_backward(const Tensor& dout, const std::vector<Tensor>& saved, int mode, bool score_before) {
  TORCH_CHECK(saved.size() == 17, "17 saved tensors expected");
  const Tensor &offs = saved[0], &src_row = saved[1], &row_score = saved[2], &pos = saved[3], &scores = saved[4],
               &h13 = saved[5];
  if (!plain(dout) || dout.scalar_type() != at::kBFloat16 || !dout.is_contiguous() || !on_current_device(dout))
    return py::none();
  for (const Tensor& t : saved)
    if (!t.is_contiguous() || t.device() != dout.device()) return py::none();
  if (h13.dim() != 3 || h13.size(0) != 2 || pos.dim() != 2 || h13.scalar_type() != at::kBFloat16 ||
      saved[16].scalar_type() != at::kBFloat16)
    return py::none();
  const int64_t T = dout.size(0), D = dout.size(1), G = offs.numel(), R = h13.size(1), H = h13.size(2), k = pos.size(1);
  const int64_t weight = G * D * H, tokens_d = up128(D) * (R / 32), tokens_h = up128(H) * (R / 32);
  const int64_t sizes[] = {G, R, R, T * k, T * k, 2 * R * H, weight, weight / 32, D * R, tokens_d, H * R, tokens_h,
                           weight, weight / 32, weight, weight / 32, (score_before ? T : R) * D};
  for (size_t i = 0; i < std::size(sizes); ++i)
    TORCH_CHECK(saved[i].numel() == sizes[i], "saved tensor ", i, " came back with ", saved[i].numel(), " elements, ",
                sizes[i], " expected");
  hipStream_t st = stream_of(dout);
  Unlocked unlocked(std::in_place);
  const int32_t* ends = offs.data_ptr<int32_t>();
  const int64_t* place = pos.data_ptr<int64_t>();
  Codes w2{saved[6], saved[7]}, xc{saved[8], saved[9]}, gc{saved[10], saved[11]}, w1{saved[12], saved[13]},
      w3{saved[14], saved[15]};
  // the casts of dout, dg, both gradients of the gate stacked (d(h1) and then d(h3)), and dx in the padded layout
  const int64_t per_r = up128(R) * (H / 32), per_c = H * (R / 32), dr_s = up128(R) * (D / 32), dc_s = D * (R / 32);
  Scratch scratch(2 * Scratch::padded(R * D) + Scratch::padded(dr_s) + Scratch::padded(dc_s) + 3 * Scratch::padded(2 * R * H) +
                      Scratch::padded(2 * per_r) + Scratch::padded(2 * per_c) + Scratch::padded(2 * R * D),
                  dout);
  const auto taken = [&](int64_t codes, int64_t scales) { return Lent{scratch.take(codes), scratch.take(scales)}; };
  const Lent dr = taken(R * D, dr_s), dc = taken(D * R, dc_s);
  checked(lib.rows_gathered(dout.data_ptr(), src_row.data_ptr<int64_t>(), score_before ? nullptr : row_score.data_ptr<float>(),
                            T, R, D, D, dr.c, dr.s, dc.c, dc.s, mode, MX_SCALES_MFMA, st),
          "mx_cast_rows_gathered");
  void* const dg = scratch.take(2 * R * H);
  checked(lib.grouped(dr.c, dr.s, w2.c(), w2.s(), ends, dg, R, H, D, G, H, MX_SCALES_MFMA, st), "mx_grouped_gemm_2d3d");
  const auto [r, rs] = taken(2 * R * H, 2 * per_r);
  const auto [c, cs] = taken(2 * H * R, 2 * per_c);
  const char* h1 = static_cast<const char*>(h13.data_ptr());
  checked(lib.swiglu_bwd_dense(dg, h1, h1 + 2 * R * H, R, H, H, H, H, r, H, rs, c, R, cs, nullptr, mode,
                               MX_SCALES_MFMA, st),
          "mx_swiglu_bwd_cast_dim0_dim1_ld");
  const Tensor dw13 = at::empty({2, G, H, D}, dout.options()), dw2 = at::empty({G, D, H}, dout.options());
  char* dw1 = static_cast<char*>(dw13.data_ptr());
  checked(lib.grouped_wgrad_two(c, cs, c + H * R, cs + per_c, xc.c(), xc.s(), ends, dw1, dw1 + 2 * G * H * D, R, H, D, G, st),
          "mx_grouped_gemm_2d2d_shared_b");
  checked(lib.grouped_wgrad(dc.c, dc.s, gc.c(), gc.s(), ends, dw2.data_ptr(), R, D, H, G, MX_SCALES_MFMA, st),
          "mx_grouped_gemm_2d2d");
  void* const dxp = scratch.take(2 * R * D);
  checked(lib.grouped_pair(r, rs, w1.c(), w1.s(), r + R * H, rs + per_r, w3.c(), w3.s(), ends, dxp, R, D, H, G, D, st),
          "mx_grouped_gemm_2d3d_pair");
  const Tensor dx = at::empty({T, D}, dout.options()), ds = at::empty({T, k}, scores.options());
  if (score_before) {
    checked(lib.combine_dot(dxp, R, D, place, scores.data_ptr<float>(), saved[16].data_ptr(), D, T, k, D,
                            dx.data_ptr(), D, ds.data_ptr<float>(), st),
            "mx_moe_combine_dot");
  } else {
    checked(lib.combine_dot(saved[16].data_ptr(), R, D, place, nullptr, dout.data_ptr(), D, T, k, D, nullptr, 0,
                            ds.data_ptr<float>(), st),
            "mx_moe_combine_dot");
    checked(lib.combine(dxp, nullptr, R, D, place, nullptr, T, k, D, dx.data_ptr(), D, st), "mx_moe_combine");
  }
  unlocked.reset();
  return py::make_tuple(dx, ds, dw13.select(0, 0), dw2, dw13.select(0, 1));
}

// ---- single launches: what the functions of ops.py of the same names do, for plain operands (else nothing)
bool matrix_of(const Tensor& t, at::ScalarType type) {
  return t.is_cuda() && t.dim() == 2 && t.scalar_type() == type && t.stride(1) == 1 && t.stride(0) >= t.size(1);
}
bool gate_rows(const Tensor& t) {
  return matrix_of(t, at::kBFloat16) && t.stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}
bool gate_sizes(int64_t T, int64_t E, int64_t D) {
  return T > 0 && E >= 8 && E <= 128 && E % 8 == 0 && D >= 128 && D % 128 == 0;
}
bool gate_grad(const Tensor& d, int64_t T, int64_t E) {
  return matrix_of(d, at::kFloat) && d.is_contiguous() && d.size(0) == T && d.size(1) == E &&
         reinterpret_cast<uintptr_t>(d.data_ptr()) % 16 == 0;
}

std::optional<Tensor> gate_logits(const Tensor& x, const Tensor& w) {
  if (!gate_rows(x) || !gate_rows(w) || x.size(1) != w.size(1) || w.device() != x.device() ||
      !gate_sizes(x.size(0), w.size(0), x.size(1)) || !on_current_device(x))
    return std::nullopt;
  const int64_t T = x.size(0), D = x.size(1), E = w.size(0);
  hipStream_t st = stream_of(x);
  Unlocked unlocked(std::in_place);
  Tensor logits = at::empty({T, E}, x.options().dtype(at::kFloat));
  checked(lib.gate_logits(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), T, E, D, logits.data_ptr<float>(), st),
          "mx_gate_logits");
  return logits;
}
std::optional<Tensor> gate_dx(const Tensor& dlogits, const Tensor& w, const std::optional<Tensor>& base) {
  if (!gate_rows(w) || dlogits.dim() != 2) return std::nullopt;
  const int64_t T = dlogits.size(0), E = w.size(0), D = w.size(1);
  if (!gate_grad(dlogits, T, E) || dlogits.device() != w.device() || !gate_sizes(T, E, D) || !on_current_device(w) ||
      (base && (!gate_rows(*base) || base->size(0) != T || base->size(1) != D || base->device() != w.device())))
    return std::nullopt;
  hipStream_t st = stream_of(w);
  Unlocked unlocked(std::in_place);
  Tensor out = at::empty({T, D}, w.options());
  checked(lib.gate_dx(dlogits.data_ptr<float>(), w.data_ptr(), w.stride(0), base ? base->data_ptr() : nullptr,
                      base ? base->stride(0) : 0, T, E, D, out.data_ptr(), st),
          "mx_gate_dx");
  return out;
}
std::optional<Tensor> gate_dw(const Tensor& dlogits, const Tensor& x) {
  if (!gate_rows(x) || dlogits.dim() != 2) return std::nullopt;
  const int64_t T = x.size(0), D = x.size(1), E = dlogits.size(1);
  if (!gate_grad(dlogits, T, E) || dlogits.device() != x.device() || !gate_sizes(T, E, D) || !on_current_device(x))
    return std::nullopt;
  hipStream_t st = stream_of(x);
  Unlocked unlocked(std::in_place);
  const Tensor work = at::empty({lib.gate_dw_workspace(T, E, D)}, x.options().dtype(at::kByte));
  Tensor out = at::empty({E, D}, x.options());
  checked(lib.gate_dw(dlogits.data_ptr<float>(), x.data_ptr(), x.stride(0), T, E, D, work.data_ptr(), out.data_ptr(), st),
          "mx_gate_dw");
  return out;
}

py::object route_topk(const Tensor& logits, const std::optional<Tensor>& bias, int64_t k, bool softmax, bool norm, double scale) {
  if (!matrix_of(logits, at::kFloat) || !logits.is_contiguous() || logits.numel() == 0 || !on_current_device(logits) ||
      (bias && (bias->scalar_type() != at::kFloat || bias->dim() != 1 || bias->size(0) != logits.size(1) ||
                !bias->is_contiguous() || bias->device() != logits.device())))
    return py::none();
  const int64_t T = logits.size(0), E = logits.size(1);
  hipStream_t st = stream_of(logits);
  Unlocked unlocked(std::in_place);
  const auto longs = logits.options().dtype(at::kLong);
  const Tensor top = at::empty({T, k}, logits.options()), selected = at::empty({T, k}, longs), counts = at::empty({E}, longs),
               block_counts = at::empty({E * ((T + 15) / 16)}, logits.options().dtype(at::kInt));
  checked(lib.route_topk(logits.data_ptr<float>(), T, E, bias ? bias->data_ptr<float>() : nullptr, k, softmax, norm,
                         static_cast<float>(scale), top.data_ptr<float>(), selected.data_ptr<int64_t>(),
                         counts.data_ptr<int64_t>(), block_counts.data_ptr<int32_t>(), st),
          "mx_route_topk");
  unlocked.reset();
  return py::make_tuple(top, selected, counts, block_counts);
}
std::optional<Tensor> route_topk_bwd(const Tensor& logits, const Tensor& selected, const Tensor& dtop, bool softmax, bool norm,
                                     double scale) {
  if (!matrix_of(logits, at::kFloat) || !logits.is_contiguous() || logits.numel() == 0 || !on_current_device(logits) ||
      selected.dim() != 2 || selected.size(0) != logits.size(0) || !plain_list(selected, at::kLong, logits) ||
      selected.sizes() != dtop.sizes() || !plain_list(dtop, at::kFloat, logits))
    return std::nullopt;
  hipStream_t st = stream_of(logits);
  Unlocked unlocked(std::in_place);
  Tensor out = at::empty(logits.sizes(), logits.options());
  checked(lib.route_topk_bwd(logits.data_ptr<float>(), logits.size(0), logits.size(1), selected.size(1), softmax, norm,
                             static_cast<float>(scale), selected.data_ptr<int64_t>(), dtop.data_ptr<float>(),
                             out.data_ptr<float>(), st),
          "mx_route_topk_bwd");
  return out;
}

py::object token_logprob_fwd(const Tensor& logits, const Tensor& target, int64_t splits) {
  if (!matrix_of(logits, at::kBFloat16) || logits.size(0) == 0 || target.dim() != 1 || target.size(0) != logits.size(0) ||
      !plain_list(target, at::kLong, logits) || !on_current_device(logits))
    return py::none();
  const int64_t rows = logits.size(0);
  hipStream_t st = stream_of(logits);
  Unlocked unlocked(std::in_place);
  const auto floats = logits.options().dtype(at::kFloat);
  const Tensor lp = at::empty({rows}, floats), lse = at::empty({rows}, floats),
               partial = splits > 1 ? at::empty({2 * rows * splits}, floats) : Tensor();
  checked(lib.logprob_fwd(logits.data_ptr(), rows, logits.size(1), logits.stride(0), target.data_ptr<int64_t>(),
                          lp.data_ptr<float>(), lse.data_ptr<float>(), splits, splits > 1 ? partial.data_ptr<float>() : nullptr,
                          st),
          "mx_token_logprob_fwd_split");
  unlocked.reset();
  return py::make_tuple(lp, lse);
}
std::optional<Tensor> token_logprob_bwd(const Tensor& logits, const Tensor& target, const Tensor& lse, const Tensor& grad) {
  if (!matrix_of(logits, at::kBFloat16) || !on_current_device(logits) || logits.size(0) == 0 || logits.size(0) > 65535)
    return std::nullopt;
  const int64_t rows = logits.size(0), vocab = logits.size(1), width = (vocab + 7) / 8 * 8;
  if (!plain_list(target, at::kLong, logits) || !plain_list(lse, at::kFloat, logits) || !plain_list(grad, at::kFloat, logits) ||
      target.numel() != rows || lse.numel() != rows || grad.numel() != rows)
    return std::nullopt;
  hipStream_t st = stream_of(logits);
  Unlocked unlocked(std::in_place);
  Tensor out = at::empty({rows, width}, logits.options());
  checked(lib.logprob_bwd(logits.data_ptr(), rows, vocab, logits.stride(0), target.data_ptr<int64_t>(), lse.data_ptr<float>(),
                          grad.data_ptr<float>(), out.data_ptr(), width, st),
          "mx_token_logprob_bwd_any");
  return vocab == width ? out : out.slice(1, 0, vocab);
}

// [(codes, scales)] of the hand-over's casts
py::object rows_many(const std::vector<Tensor>& tensors, int mode) {
  const size_t n = tensors.size();
  for (const Tensor& t : tensors)
    if (!t.is_cuda() || t.device() != tensors[0].device() || !on_current_device(t) || !t.is_contiguous() || t.dim() == 0 ||
        (t.scalar_type() != at::kBFloat16 && t.scalar_type() != at::kFloat) || t.numel() == 0 || t.size(-1) % 32 ||
        reinterpret_cast<uintptr_t>(t.data_ptr()) % 16)
      return py::none();
  if (n == 0) return py::none();
  hipStream_t st = stream_of(tensors[0]);
  std::vector<std::pair<Tensor, Tensor>> out(n);
  {
    Unlocked unlocked(std::in_place);
    std::vector<const void*> x(n);
    std::vector<int64_t> elems(n);
    std::vector<int32_t> f32(n);
    std::vector<uint8_t*> codes(n), scales(n);
    for (size_t i = 0; i < n; ++i) {
      const Tensor& t = tensors[i];
      const auto bytes = at::TensorOptions().device(t.device()).dtype(at::kByte);
      std::vector<int64_t> sizes = t.sizes().vec();
      out[i].first = at::empty(sizes, bytes);
      sizes.back() /= 32;
      out[i].second = at::empty(sizes, bytes);
      x[i] = t.data_ptr();
      elems[i] = t.numel();
      f32[i] = t.scalar_type() == at::kFloat;
      codes[i] = out[i].first.data_ptr<uint8_t>();
      scales[i] = out[i].second.data_ptr<uint8_t>();
    }
    checked(lib.rows_many(n, x.data(), elems.data(), f32.data(), codes.data(), scales.data(), mode, st), "mx_cast_rows_many");
  }
  return py::cast(out);
}
std::optional<std::vector<Tensor>> dequant_many(const std::vector<Tensor>& codes, const std::vector<Tensor>& scales) {
  const size_t n = codes.size();
  if (n == 0 || scales.size() != n) return std::nullopt;
  for (size_t i = 0; i < n; ++i) {
    const Tensor &c = codes[i], &s = scales[i];
    if (!c.is_cuda() || c.device() != codes[0].device() || s.device() != c.device() || !on_current_device(c) || c.dim() == 0 ||
        !c.is_contiguous() || !s.is_contiguous() || c.scalar_type() != at::kByte || s.scalar_type() != at::kByte ||
        c.numel() == 0 || c.size(-1) % 32 || s.numel() * 32 != c.numel())
      return std::nullopt;
  }
  hipStream_t st = stream_of(codes[0]);
  Unlocked unlocked(std::in_place);
  std::vector<const uint8_t*> c(n), s(n);
  std::vector<int64_t> elems(n);
  std::vector<void*> to(n);
  std::vector<Tensor> out(n);
  for (size_t i = 0; i < n; ++i) {
    out[i] = at::empty(codes[i].sizes(), at::TensorOptions().device(codes[i].device()).dtype(at::kBFloat16));
    c[i] = codes[i].data_ptr<uint8_t>();
    s[i] = scales[i].data_ptr<uint8_t>();
    elems[i] = codes[i].numel();
    to[i] = out[i].data_ptr();
  }
  checked(lib.dequant_many(n, c.data(), s.data(), elems.data(), to.data(), st), "mx_dequant_many");
  return out;
}

// The capture that `stream` is part of, a number of its own for every capture (0: none).
unsigned long long capture_id(uintptr_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  const hipError_t rc = hipStreamGetCaptureInfo(reinterpret_cast<hipStream_t>(stream), &status, &id);
  TORCH_CHECK(rc == hipSuccess, "hipStreamGetCaptureInfo: ", hipGetErrorString(rc));
  return status == hipStreamCaptureStatusNone ? 0 : id;
}

}  // namespace

// (errors of torch keep their types: an allocation that fails is a torch.OutOfMemoryError)
PYBIND11_MODULE(_blocks, m) {
  m.def("bind", &bind);
  m.def("capture_id", torch::wrap_pybind_function(capture_id));
  m.def("linear_forward", torch::wrap_pybind_function(linear_forward));
  m.def("linear_backward", torch::wrap_pybind_function(linear_backward));
  m.def("linear_apply", torch::wrap_pybind_function(linear_apply));
  m.def("ffn_forward", torch::wrap_pybind_function(ffn_forward));
  m.def("ffn_backward", torch::wrap_pybind_function(ffn_backward));
  m.def("routed_forward", torch::wrap_pybind_function(routed_forward));
  m.def("routed_backward", torch::wrap_pybind_function(routed_backward));
  m.def("gate_logits", torch::wrap_pybind_function(gate_logits));
  m.def("gate_dx", torch::wrap_pybind_function(gate_dx));
  m.def("gate_dw", torch::wrap_pybind_function(gate_dw));
  m.def("route_topk", torch::wrap_pybind_function(route_topk));
  m.def("route_topk_bwd", torch::wrap_pybind_function(route_topk_bwd));
  m.def("token_logprob_fwd", torch::wrap_pybind_function(token_logprob_fwd));
  m.def("token_logprob_bwd", torch::wrap_pybind_function(token_logprob_bwd));
  m.def("rows_many", torch::wrap_pybind_function(rows_many));
  m.def("dequant_many", torch::wrap_pybind_function(dequant_many));
}
