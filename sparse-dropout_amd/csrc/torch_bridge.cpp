// The autograd side of the package in native code: one Python call per layer (or stack) and direction instead of a
// Python autograd function around ctypes calls.
//
// What bounds a step of a small layer is the host: at 128 x 256 -> 256 the two launches of a step run for 19 us and
// the Python path around them (argument checks, tensor views, 45-argument ctypes calls, the backward's hop into the
// interpreter on autograd's thread) took 64-146 us, depending on the host.  Here the checks, the allocations, the
// library calls and the backward node are compiled, and the backward runs without the interpreter lock.
//
// Every computation is a call into libsparsedrop.so through its C ABI; torch owns memory, streams and the graph.
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/extension.h>

#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <array>
#include <atomic>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "sparsedrop.h"

#if __has_include("source_hash.inc")
#include "source_hash.inc"
#else
#define SD_SOURCE_HASH "unknown"
#endif

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

PyObject* library_error = nullptr;  // SparseDropError, once the loader has handed it over

// Raised on whatever thread a call failed on (a backward runs on autograd's), so with the interpreter lock taken.
[[noreturn]] void raise_library_error(const std::string& msg) {
  pybind11::gil_scoped_acquire gil;
  PyErr_SetString(library_error ? library_error : PyExc_RuntimeError, msg.c_str());
  python_error err;
  err.persist();
  throw std::move(err);
}

void check(int rc, const char* fn) {
  if (rc == SD_OK) return;
  const std::string msg = std::string(fn) + ": " + sd_last_error();
  TORCH_CHECK_VALUE(rc != SD_ERR_INVALID, msg);
  TORCH_CHECK_NOT_IMPLEMENTED(rc != SD_ERR_UNSUPPORTED, msg);
  raise_library_error(msg);
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

int dtype_of(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? SD_BF16 : SD_F16; }

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// ---- operands -----------------------------------------------------------------------------------------------------
// `x` itself when it is a row- or column-major matrix in memory, else a contiguous copy (expanded or doubly strided).
Tensor as_matrix(const Tensor& x) {
  const int64_t rows = x.size(0), cols = x.size(1), sr = x.stride(0), sc = x.stride(1);
  if (sc == 1 && (rows <= 1 || sr >= cols)) return x;
  if (sr == 1 && (cols <= 1 || sc >= rows)) return x;
  return x.contiguous();
}

// pointer and element strides; the stride of an extent-1 dimension is arbitrary in torch and normalised here
struct Mat {
  void* ptr = nullptr;
  int64_t sr = 0, sc = 0;
  Mat() = default;
  explicit Mat(const Tensor& t) : ptr(t.data_ptr()), sr(t.stride(0)), sc(t.stride(1)) {
    const int64_t rows = t.size(0), cols = t.size(1);
    if (rows <= 1 && sc == 1) sr = std::max<int64_t>(cols, 1);
    if (cols <= 1 && sr == 1) sc = std::max<int64_t>(rows, 1);
    sr = std::max<int64_t>(sr, 1);
    sc = std::max<int64_t>(sc, 1);
  }
};
#define MAT(m) (m).ptr, (m).sr, (m).sc

void check_operand(const char* name, const Tensor& x) {
  TORCH_CHECK_VALUE(x.is_cuda(), name, " must be on the GPU (got ", x.device(), ")");
  TORCH_CHECK_VALUE(x.dim() == 2, name, " must be 2D (got ", x.dim(), "D)");
  TORCH_CHECK_TYPE(x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16, name,
                   " must be float16 or bfloat16 (got ", x.dtype(), ")");
  TORCH_CHECK_VALUE(x.numel() == 0 || x.stride(0) == 1 || x.stride(1) == 1, name,
                    " must be row or column major (strides ", x.strides(), ")");
}

void check_pair(const Tensor& a, const Tensor& b) {
  check_operand("A", a);
  check_operand("B", b);
  TORCH_CHECK_TYPE(a.scalar_type() == b.scalar_type(), "A and B must have the same dtype (", a.dtype(), " vs ",
                   b.dtype(), ")");
  TORCH_CHECK_VALUE(a.device() == b.device(), "A and B must be on the same device");
  TORCH_CHECK_VALUE(a.size(1) == b.size(1), "reduction dims differ: A ", a.sizes(), ", B ", b.sizes());
}

// The mask itself when it is row- or column-major in memory, else (expanded: stride 0, or doubly strided) a copy.
Tensor check_mask(const Tensor& mask, int64_t mb, int64_t kb, const Tensor& like) {
  TORCH_CHECK_TYPE(mask.scalar_type() == at::kBool, "Mask must be bool (got ", mask.dtype(), ")");
  TORCH_CHECK_VALUE(mask.device() == like.device(), "mask must be on the same device as the operands");
  TORCH_CHECK_VALUE(mask.dim() == 2 && mask.size(0) == mb && mask.size(1) == kb, "mask shape ", mask.sizes(),
                    " does not match blocks [", mb, ", ", kb, "]");
  const bool expanded = (mb > 1 && mask.stride(0) == 0) || (kb > 1 && mask.stride(1) == 0);
  return expanded || (mask.stride(0) != 1 && mask.stride(1) != 1) ? mask.contiguous() : mask;
}

struct MaskArg {
  const uint8_t* ptr = nullptr;
  int64_t sr = 0, sc = 0;
  MaskArg() = default;
  explicit MaskArg(const Tensor& m) : ptr(static_cast<const uint8_t*>(m.data_ptr())), sr(m.stride(0)), sc(m.stride(1)) {
    if (sr != 1 && sc != 1) {  // only possible for degenerate shapes
      sr = m.size(1);
      sc = 1;
    }
    sr = std::max<int64_t>(sr, 1);  // (of an extent of 1: no stride over more is 0 here)
    sc = std::max<int64_t>(sc, 1);
  }
};

Tensor new_matrix(const Tensor& like, int64_t rows, int64_t cols) { return at::empty({rows, cols}, like.options()); }

// ---- operands whose rows do not start on 16-byte boundaries -----------------------------------------------------------
// An odd width (or a slice that starts off a boundary) would put 16-byte loads across row ends.  Copies with padded rows
// keep such products on the specialised kernels: the columns and rows added are zeros, so every sum is unchanged, and
// extents that only bound a result stay what they were.  Up to four operands share a launch.  A step
// of 3001 x 1025 -> 777 (bf16, p = 0.3): 310 us on the kernel that takes any layout, 66 with the copies.
bool row_major(const Tensor& t) { return Mat(t).sc == 1; }
bool rows_on_16_bytes(const Tensor& t) {
  return Mat(t).sr % 8 == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

struct RowPadding {
  int n = 0;
  const void* src[4];
  void* dst[4];
  int64_t ld[4], rows[4], cols[4], dst_rows[4], dst_ld[4];
  std::vector<Tensor> keep;  // the sources, which may be contiguous copies made here
  // a [rows_out, width rounded up to 8] copy of t, filled by launch()
  Tensor add(const Tensor& t_, int64_t rows_out) {
    const Tensor t = row_major(t_) ? t_ : t_.contiguous();
    keep.push_back(t);
    const Mat m(t);
    const int64_t width = ceil_div(t.size(1), 8) * 8;
    Tensor out = new_matrix(t, rows_out, width);
    src[n] = m.ptr;
    ld[n] = m.sr;
    rows[n] = t.size(0);
    cols[n] = t.size(1);
    dst[n] = out.data_ptr();
    dst_rows[n] = rows_out;
    dst_ld[n] = width;
    ++n;
    return out;
  }
  void launch() {
    if (n == 0) return;
    c10::DeviceGuard guard(keep[0].device());
    check(sd_pad_rows(n, src, ld, rows, cols, dst, dst_rows, dst_ld, stream_of(keep[0])), "sd_pad_rows");
  }
};

// Operands of A . B^T (both row-major, the width is the reduction) with padded rows where they need it.
void pad_reduction(Tensor& a, Tensor& b) {
  const int64_t K = a.size(1);
  if (a.size(0) == 0 || b.size(0) == 0 || K == 0 || !row_major(a) || !row_major(b)) return;
  RowPadding pad;
  if (K % 8 || !rows_on_16_bytes(a)) a = pad.add(a, a.size(0));
  if (K % 8 || !rows_on_16_bytes(b)) b = pad.add(b, b.size(0));
  pad.launch();
}

// fp32 scratch for a split reduction, when the library wants one for this shape
struct Scratch {
  Tensor t;
  void* ptr = nullptr;
  int64_t bytes = 0;
  Scratch(const Tensor& like, int64_t nbytes) {
    if (nbytes <= 0) return;
    t = at::empty({nbytes / 4}, like.options().dtype(at::kFloat));
    ptr = t.data_ptr();
    bytes = nbytes;
  }
};

// ---- mask and kept-block lists of one layer ---------------------------------------------------------------------------
// One int32 buffer: row_ptr | col_ptr | col_idx | row_idx | bytes of a drawn mask.  `given` keeps a caller's mask alive.
struct Lists {
  Tensor buf, given;
  int64_t bs = 0;         // block size of the mask
  int64_t kernel_bs = 0;  // what the list-taking calls are told: 64, or 32 when the lists carry quadrant bits
  int64_t mb = 0, kb = 0;          // mask grid
  int64_t out_mb = 0, out_kb = 0;  // listed grid
  bool mask_only = false;          // no lists: the buffer holds a drawn mask or nothing

  void shape(int64_t rows, int64_t cols, int64_t bs_) {
    bs = bs_;
    const int64_t g = bs % 32 == 0 ? 64 : bs;
    kernel_bs = bs % 64 == 32 ? 32 : g;
    mb = ceil_div(rows, bs);
    kb = ceil_div(cols, bs);
    out_mb = ceil_div(rows, g);
    out_kb = ceil_div(cols, g);
    TORCH_CHECK_VALUE(mb > 0 && kb > 0, "mask must be non-empty");
  }
  void allocate(const Tensor& like, const OptTensor& mask) {
    if (mask) given = check_mask(*mask, mb, kb, like);
    const int64_t ints = (mask_only ? 0 : out_mb + out_kb + 2 + 2 * out_mb * out_kb) + (mask ? 0 : (mb * kb + 3) / 4);
    buf = at::empty({ints}, like.options().dtype(at::kInt));
  }
  int32_t* row_ptr() const { return static_cast<int32_t*>(buf.data_ptr()); }
  int32_t* col_ptr() const { return row_ptr() + out_mb + 1; }
  int32_t* col_idx() const { return col_ptr() + out_kb + 1; }
  int32_t* row_idx() const { return col_idx() + out_mb * out_kb; }
  uint8_t* drawn() const {
    return given.defined() ? nullptr : reinterpret_cast<uint8_t*>(mask_only ? row_ptr() : row_idx() + out_mb * out_kb);
  }
  MaskArg mask() const {
    if (given.defined()) return MaskArg(given);
    MaskArg m;
    m.ptr = drawn();
    m.sr = kb;
    m.sc = 1;
    return m;
  }
};

// ---- what a node keeps for its backward ----------------------------------------------------------------------------------
// A tensor that goes through torch's saved-tensor hooks (offloading and checkpoints take its memory in between) and is
// checked for writes since it was saved.  A hook may hand back any tensor, and the launches trust pointers and extents:
// what comes back has to have the type, device and extents of what was saved; its strides may be others.
struct Saved {
  SavedVariable tensor;
  at::DimVector sizes;
  at::ScalarType dtype = at::kHalf;
  c10::Device device = c10::Device(at::kCPU);
  void keep(const Tensor& t) {
    if (!t.defined()) return;
    tensor = SavedVariable(t, false);
    sizes = t.sizes();
    dtype = t.scalar_type();
    device = t.device();
  }
  Tensor get() const {  // undefined when nothing was kept
    Tensor t = tensor.unpack();
    TORCH_CHECK_VALUE(!t.defined() || (t.sizes() == at::IntArrayRef(sizes) && t.scalar_type() == dtype && t.device() == device),
                      "a saved-tensor hook returned a ", t.sizes(), " ", t.dtype(), " tensor on ", t.device(), " for a ",
                      at::IntArrayRef(sizes), " ", dtype, " tensor on ", device);
    return t;
  }
  Tensor matrix() const {
    const Tensor t = get();
    return t.defined() ? as_matrix(t) : t;
  }
  void drop() { tensor.reset_data(); }
};

struct SavedLists {
  Saved buf, given;
  Lists shape;  // without its tensors
  // mask: the tensor whose changes count, when that is not the one in the lists
  void keep(Lists&& lists, const Tensor& mask = Tensor()) {
    buf.keep(lists.buf);
    given.keep(mask.defined() ? mask : lists.given);
    shape = std::move(lists);
    shape.buf.reset();
    shape.given.reset();
  }
  Lists get() const {  // undefined buffer: no lists were made
    Lists l = shape;
    l.buf = buf.get();
    if (l.buf.defined()) l.buf = l.buf.contiguous();
    const Tensor mask = given.get();
    if (mask.defined()) l.given = check_mask(mask, l.mb, l.kb, mask);
    return l;
  }
  void drop() {
    buf.drop();
    given.drop();
  }
};

// Where a layer's mask comes from: given, pinned by a seed, or from the device-resident generator state.
struct Draw {
  OptTensor mask;
  std::optional<uint64_t> seed;
  OptTensor state;
  uint64_t* state_ptr() const {
    return (mask || seed || !state) ? nullptr : static_cast<uint64_t*>(state->data_ptr());
  }
};

void check_p(double p) { TORCH_CHECK_VALUE(p >= 0.0 && p < 1.0, "p must be in [0, 1), got ", p); }

// ---- the products of one layer ----------------------------------------------------------------------------------------
// Y = act(s (keep . X) W^T) with mask and lists, one library call; pre: receives the pre-activation when wanted.
// drawn: the lists are allocated and hold a drawn mask, and `draw` isn't asked.
Tensor layer_forward(Tensor x, Tensor w, int64_t bs, double p, const Draw& draw, int act, bool want_pre, Lists& lists,
                     Tensor* pre, bool drawn = false) {
  check_pair(x, w);
  check_p(p);
  lists.shape(x.size(0), x.size(1), bs);
  if (bs % 32 == 0) pad_reduction(x, w);  // (a width rounded up to 8 has the same block grid)
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  if (!drawn) lists.allocate(x, draw.mask);
  Tensor y = new_matrix(x, M, N);
  if (want_pre && act != SD_ACT_NONE) *pre = new_matrix(x, M, N);
  const int64_t g = bs % 32 == 0 ? 64 : bs;
  Scratch ws(x, sd_splitk_workspace_bytes(M, N, K, g, 1));
  const MaskArg given = draw.mask || drawn ? lists.mask() : MaskArg();
  Mat pm;
  if (pre && pre->defined()) pm = Mat(*pre);
  const Mat xm(x), wm(w), ym(y);
  c10::DeviceGuard guard(x.device());
  check(sd_dropout_matmul_forward_act(MAT(xm), MAT(wm), MAT(ym), given.ptr, given.sr, given.sc,
                                      drawn ? nullptr : draw.state_ptr(), draw.seed.value_or(0), 0, p,
                                      drawn ? nullptr : lists.drawn(), lists.row_ptr(), lists.col_idx(), lists.col_ptr(),
                                      lists.row_idx(), M, N, K, bs, dtype_of(x), act, MAT(pm), ws.ptr, ws.bytes, stream_of(x)),
        "sd_dropout_matmul_forward_act");
  return y;
}

// dX and / or dW of one layer in one library call; act_at: what dX's fused activation derivative is evaluated at.
// kept_only (without an activation): dropped blocks of dX are left as they are.
std::pair<Tensor, Tensor> layer_products(const Tensor& dy, const Tensor& w, const Tensor& x, const Lists& lists, double p,
                                         bool need_dx, bool need_dw, int act, const Tensor& act_at, bool kept_only = false) {
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  Tensor dx = need_dx ? new_matrix(x, M, K) : Tensor(), dw = need_dw ? new_matrix(x, N, K) : Tensor();
  if (!(need_dx || need_dw) || M == 0 || K == 0) return {dx, dw};
  if (N == 0) return {need_dx ? dx.zero_() : dx, dw};
  const int64_t g = lists.kernel_bs == 32 ? 64 : lists.kernel_bs;
  Scratch ws(x, need_dw ? sd_splitk_workspace_bytes(K, N, M, g, 1) : 0);
  if (!need_dx) act = SD_ACT_NONE;
  Mat am, dxm, dwm;
  if (act != SD_ACT_NONE) am = Mat(act_at);
  if (need_dx) dxm = Mat(dx);
  if (need_dw) dwm = Mat(dw);
  const Mat gm(dy), wm(w), xm(x);
  c10::DeviceGuard guard(x.device());
  if (kept_only) {
    check(sd_dropout_matmul_backward_kept(MAT(gm), MAT(wm), MAT(xm), MAT(dxm), MAT(dwm), lists.row_ptr(), lists.col_idx(),
                                          lists.col_ptr(), lists.row_idx(), M, N, K, lists.kernel_bs, p, dtype_of(x), ws.ptr,
                                          ws.bytes, stream_of(x)),
          "sd_dropout_matmul_backward_kept");
    return {dx, dw};
  }
  check(sd_dropout_matmul_backward_act(MAT(gm), MAT(wm), MAT(xm), MAT(dxm), MAT(dwm), lists.row_ptr(), lists.col_idx(),
                                       lists.col_ptr(), lists.row_idx(), M, N, K, lists.kernel_bs, p, dtype_of(x), act,
                                       MAT(am), ws.ptr, ws.bytes, stream_of(x)),
        "sd_dropout_matmul_backward_act");
  return {dx, dw};
}

// The same for gradients and operands of any width.
std::pair<Tensor, Tensor> layer_backward(const Tensor& dy, const Tensor& w, const Tensor& x, const Lists& lists,
                                         double p, bool need_dx, bool need_dw, int act, const Tensor& act_at) {
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK_VALUE(dy.size(0) == M && dy.size(1) == N && dy.device() == x.device(), "dy must be a [", M, ", ", N,
                    "] tensor on ", x.device());
  if (N > 0 && M > 0 && K > 0 && (need_dx || need_dw)) {
    // dY's width is a reduction (dX) and so is W's height: zero columns and rows up to the next multiple of 8 (the
    // reference pads a 10-class head to 128 outputs up front, eval/mlp/model.py:22-24,40); dX is unchanged and the extra
    // rows of dW are dropped.  X and the width of W only need rows on 16-byte boundaries.
    const int64_t n8 = ceil_div(N, 8) * 8;
    const bool rows = row_major(dy) && (!need_dx || row_major(w)) && (!need_dw || row_major(x));
    const bool pad_dy = N % 8 || (rows && !rows_on_16_bytes(dy));
    const bool pad_w = need_dx && (N % 8 || (rows && !rows_on_16_bytes(w)));
    const bool pad_x = need_dw && rows && !rows_on_16_bytes(x);
    if (pad_dy || pad_w || pad_x) {
      RowPadding pad;
      Tensor dyp = dy, wp = w, xp = x;
      if (pad_dy) dyp = pad.add(dy, M);
      if (pad_w) wp = pad.add(w, n8).narrow(1, 0, K);
      else if (N % 8) wp = at::empty({n8, K}, w.options());  // dW alone: only its shape is looked at
      if (pad_x) xp = pad.add(x, M).narrow(1, 0, K);
      pad.launch();
      auto [dx, dw] = layer_products(dyp, wp, xp, lists, p, need_dx, need_dw, act, act_at);
      return {dx, dw.defined() && n8 != N ? dw.narrow(0, 0, N) : dw};
    }
  }
  return layer_products(dy, w, x, lists, p, need_dx, need_dw, act, act_at);
}

// A . B^T without dropout, with the activation in the store.
Tensor dense(Tensor a, Tensor b, int act, bool want_pre, Tensor* pre) {
  check_pair(a, b);
  pad_reduction(a, b);
  const int64_t M = a.size(0), N = b.size(0), K = a.size(1);
  Tensor c = new_matrix(a, M, N);
  if (want_pre && act != SD_ACT_NONE) *pre = new_matrix(a, M, N);
  if (M == 0 || N == 0) return c;
  Mat pm;
  if (pre && pre->defined()) {
    pm = Mat(*pre);
    if (K == 0) pre->zero_();
  }
  if (K == 0) return c.zero_();
  Scratch ws(a, sd_splitk_workspace_bytes(M, N, K, 0, 0));
  const Mat am(a), bm(b), cm(c);
  c10::DeviceGuard guard(a.device());
  check(sd_gemm_act(MAT(am), MAT(bm), MAT(cm), M, N, K, dtype_of(a), act, MAT(pm), ws.ptr, ws.bytes, stream_of(a)),
        "sd_gemm_act");
  return c;
}

Tensor grad_matrix(const Tensor& g, const Tensor& like) {
  return as_matrix(g.scalar_type() == like.scalar_type() ? g : g.to(like.scalar_type()));
}

template <typename N>
bool records(const N& inputs) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor& t : inputs)
    if (t.requires_grad()) return true;
  return false;
}

// There is no forward-mode formula, and the launches read the primal values only: an input that carries a forward gradient
// would silently lose it.
template <typename N>
void refuse_forward_mode(const N& inputs) {
  for (const Tensor& t : inputs)
    TORCH_CHECK_NOT_IMPLEMENTED(!torch::autograd::isFwGradDefined(t), "block dropout products have no jvp: forward mode AD is "
                                "not supported");
}

// A product computed without recording; the node is attached to its result afterwards.
struct NoRecord {
  at::AutoDispatchBelowADInplaceOrView below;
};

// Autocast contract of the reference (custom_fwd(cast_inputs=torch.float16), blockwise_dropout_matmul_cuda.py:9): under
// autocast the operands are cast to the autocast dtype; outside it they must already be float16 / bfloat16.
Tensor autocast(const Tensor& t) {
  return at::autocast::is_autocast_enabled(at::kCUDA) ? t.to(at::autocast::get_autocast_dtype(at::kCUDA)) : t;
}

// A gradient that is not there (a function behind the output returned none) counts as zeros in the nodes below, as it does
// in Python autograd functions: the parameters get a gradient of zeros, not none.

// ---- one layer ----------------------------------------------------------------------------------------------------------
struct LinearBackward : Node {
  Saved x, w;
  SavedLists lists;
  double p = 0;
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    at::NoGradGuard no_grad;
    variable_list out(2);
    const Tensor xs = x.matrix(), ws = w.matrix();
    const Tensor dy = grads[0].defined() ? grad_matrix(grads[0], xs) : at::zeros({xs.size(0), ws.size(0)}, xs.options());
    const bool need_dx = task_should_compute_output(0), need_dw = task_should_compute_output(1);
    std::tie(out[0], out[1]) = layer_backward(dy, ws, xs, lists.get(), p, need_dx, need_dw, SD_ACT_NONE, Tensor());
    return out;
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    x.drop();
    w.drop();
    lists.drop();
  }
  std::string name() const override { return "BlockwiseDropoutMatmulHIPBackward"; }
};

template <typename B>
std::shared_ptr<B> make_node(const variable_list& inputs) {
  std::shared_ptr<B> node(new B(), torch::autograd::deleteNode);
  node->set_next_edges(torch::autograd::collect_next_edges(inputs));
  return node;
}

Tensor linear(const Tensor& input, const Tensor& weight, const OptTensor& mask, int64_t bs, double p,
              std::optional<uint64_t> seed, const OptTensor& state) {
  TORCH_CHECK_VALUE(input.dim() == 2 && weight.dim() == 2, "input must be [M, K] and weight [N, K]");
  const Tensor x = as_matrix(autocast(input)), w = as_matrix(autocast(weight));
  refuse_forward_mode(std::array<Tensor, 2>{x, w});
  Lists lists;
  Tensor y;
  {
    NoRecord guard;
    y = layer_forward(x, w, bs, p, Draw{mask, seed, state}, SD_ACT_NONE, false, lists, nullptr);
  }
  if (records(std::array<Tensor, 2>{x, w})) {
    auto node = make_node<LinearBackward>({x, w});
    node->x.keep(x);
    node->w.keep(w);
    node->lists.keep(std::move(lists));
    node->p = p;
    torch::autograd::set_history(y, node);
  }
  return y;
}

// ---- a stack of layers with an activation between consecutive ones -------------------------------------------------------
// (see functional/blockwise_dropout_mlp_hip.py for what is computed)
struct MlpBackward : Node {
  Saved x;
  std::vector<Saved> ws;
  std::vector<Saved> hidden, pre;  // activated outputs of all layers but the last; GELU: their pre-activations
  std::vector<SavedLists> lists;   // nothing kept: the layer ran dense
  std::vector<double> ps;
  int act = SD_ACT_NONE;
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    at::NoGradGuard no_grad;
    const int n = (int)ws.size();
    variable_list out(1 + n);
    const Tensor x0 = x.matrix();
    Tensor g = grads[0].defined() ? grad_matrix(grads[0], x0) : at::zeros({x0.size(0), ws.back().sizes[0]}, x0.options());
    for (int i = n - 1; i >= 0; --i) {
      const Tensor w = ws[i].matrix(), h = i ? hidden[i - 1].matrix() : x0;
      const Lists l = lists[i].get();
      const bool need_w = task_should_compute_output(1 + i), need_in = i > 0 || task_should_compute_output(0);
      if (!l.buf.defined()) {  // the dense first layer: only its weight gradient is wanted, dW = g^T . h
        if (need_w) {
          const int64_t N = w.size(0);
          Tensor gp = g, hp = h;
          const bool some = g.size(0) > 0 && N > 0 && h.size(1) > 0, rows = some && row_major(g) && row_major(h);
          RowPadding pad;
          if (some && (N % 8 || (rows && !rows_on_16_bytes(g)))) gp = pad.add(g, g.size(0));
          if (rows && !rows_on_16_bytes(h)) hp = pad.add(h, h.size(0)).narrow(1, 0, h.size(1));
          pad.launch();
          const Tensor dw = dense(gp.t(), hp.t(), SD_ACT_NONE, false, nullptr);
          out[1 + i] = dw.size(0) != N ? dw.narrow(0, 0, N) : dw;
        }
        break;
      }
      Tensor at;
      if (i > 0 && need_in && act != SD_ACT_NONE) at = act == SD_ACT_GELU ? pre[i - 1].matrix() : h;
      // both gradients of the layer in one library call, the activation's derivative riding on the dX store
      auto [dx, dw] = layer_backward(g, w, h, l, ps[i], need_in, need_w, at.defined() ? act : SD_ACT_NONE, at);
      out[1 + i] = dw;
      if (!need_in) break;
      g = dx;
      if (i == 0) out[0] = dx;
    }
    return out;
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    x.drop();
    for (auto* saved : {&ws, &hidden, &pre})
      for (Saved& s : *saved) s.drop();
    for (SavedLists& l : lists) l.drop();
  }
  std::string name() const override { return "BlockwiseDropoutMLPHIPBackward"; }
};

Tensor mlp(const Tensor& input, const std::vector<Tensor>& weights, int64_t bs, const std::vector<double>& ps, int act,
           const std::optional<std::vector<OptTensor>>& masks, std::optional<uint64_t> seed, const OptTensor& state) {
  const int n = (int)weights.size();
  bool two_d = input.dim() == 2;
  for (const Tensor& w : weights) two_d = two_d && w.dim() == 2;
  TORCH_CHECK_VALUE(two_d, "input must be [M, K] and every weight [out, in]");
  const Tensor x = as_matrix(autocast(input));
  std::vector<Tensor> ws;
  ws.reserve(n);
  for (const Tensor& w : weights) ws.push_back(as_matrix(autocast(w)));
  variable_list inputs{x};
  inputs.insert(inputs.end(), ws.begin(), ws.end());
  refuse_forward_mode(inputs);
  const bool rec = records(inputs);
  // (whether it is recorded or not: which of the generator's draws a layer takes does not depend on the gradient mode)
  const bool x_grad = x.requires_grad();
  std::vector<Lists> lists(n);
  std::vector<Tensor> hidden, pres;
  Tensor h = x;
  {
    NoRecord guard;
    for (int i = 0; i < n; ++i) {
      const bool last = i + 1 == n;
      const int a = last ? SD_ACT_NONE : act;
      const bool want_pre = a == SD_ACT_GELU && rec;
      Tensor pre, out;
      if (i == 0 && ps[0] == 0.0 && !masks && !x_grad) {
        // a first layer without dropout whose input needs no gradient (the reference's models start with one,
        // eval/mlp/model.py:31-33): the dense product with the same fused store, no mask and no lists
        out = dense(h, ws[0], a, want_pre, &pre);
      } else {
        Draw draw{masks ? (*masks)[i] : OptTensor(),
                  seed ? std::optional<uint64_t>(*seed + (uint64_t)i) : std::nullopt, state};
        out = layer_forward(h, ws[i], bs, ps[i], draw, a, want_pre, lists[i], &pre);
      }
      if (!last) {
        hidden.push_back(out);
        pres.push_back(pre);
      }
      h = out;
    }
  }
  if (rec) {
    auto node = make_node<MlpBackward>(inputs);
    node->x.keep(x);
    node->ws.resize(n);
    node->hidden.resize(n - 1);
    node->pre.resize(n - 1);
    node->lists.resize(n);
    for (int i = 0; i < n; ++i) {
      node->ws[i].keep(ws[i]);
      node->lists[i].keep(std::move(lists[i]));
      if (i + 1 == n) break;
      node->hidden[i].keep(hidden[i]);
      node->pre[i].keep(pres[i]);
    }
    node->ps = ps;
    node->act = act;
    torch::autograd::set_history(h, node);
  }
  return h;
}

// ---- convolution --------------------------------------------------------------------------------------------------------
// (see functional/im2col_conv2d.py for what is computed)
// Which route each product of the process's last convolution took; 0 = not computed.
enum Route { kNone = 0, kImplicit = 1, kFused = 2, kExplicit = 3 };
std::atomic<int> last_routes[3];  // forward, dx, dw

struct ConvGeom {
  int64_t n, c, h, w, k, r, s, pad[2], stride[2], dil[2], po, qo;
  int64_t rows() const { return n * po * qo; }
  int64_t cols() const { return c * r * s; }
};
#define GEOM_X(g) (g).n, (g).c, (g).h, (g).w
#define GEOM_W(g) (g).pad[0], (g).pad[1], (g).stride[0], (g).stride[1], (g).dil[0], (g).dil[1]
#define STRIDES4(t) (t).stride(0), (t).stride(1), (t).stride(2), (t).stride(3)

void check_conv_mask(const ConvGeom& g, int64_t bs, double p, const Draw& draw, Lists& l) {
  check_p(p);
  TORCH_CHECK_VALUE(draw.mask || (float)p < 1.f, "p must be in [0, 1) in 32 bits to draw a mask, got ", p);  // whichever launch draws
  l.shape(g.rows(), g.cols(), bs);
  if (draw.mask)
    TORCH_CHECK_VALUE(draw.mask->dim() == 2 && draw.mask->size(0) == l.mb && draw.mask->size(1) == l.kb, "mask shape ",
                      draw.mask->sizes(), " != [", l.mb, ", ", l.kb, "] for a [", g.rows(), ", ", g.cols(),
                      "] matrix in blocks of ", bs);
}
void conv_mask(const Tensor& x, const ConvGeom& g, int64_t bs, double p, const Draw& draw, Lists& l) {
  check_conv_mask(g, bs, p, draw, l);
  l.allocate(x, draw.mask);
}

void conv_lists(const Tensor& x, const ConvGeom& g, int64_t bs, double p, const Draw& draw, Lists& l) {
  conv_mask(x, g, bs, p, draw, l);
  const int64_t split = bs / 64;
  c10::DeviceGuard guard(x.device());
  if (draw.mask) {
    const MaskArg m = l.mask();
    check(sd_build_lists_split(m.ptr, l.mb, l.kb, m.sr, m.sc, split, l.out_mb, l.out_kb, l.row_ptr(), l.col_idx(),
                               l.col_ptr(), l.row_idx(), stream_of(x)),
          "sd_build_lists_split");
  } else if (uint64_t* st = draw.state_ptr()) {
    check(sd_random_lists_state(st, (float)p, l.mb, l.kb, l.drawn(), split, l.out_mb, l.out_kb, l.row_ptr(),
                                l.col_idx(), l.col_ptr(), l.row_idx(), stream_of(x)),
          "sd_random_lists_state");
  } else {
    check(sd_random_lists(draw.seed.value_or(0), 0, (float)p, l.mb, l.kb, l.drawn(), split, l.out_mb, l.out_kb,
                          l.row_ptr(), l.col_idx(), l.col_ptr(), l.row_idx(), stream_of(x)),
          "sd_random_lists");
  }
}

// A 1 x 1 kernel that visits every pixel once: the patch matrix is the image's pixels as rows.
bool pointwise(const ConvGeom& g) {
  return g.r == 1 && g.s == 1 && g.pad[0] == 0 && g.pad[1] == 0 && g.stride[0] == 1 && g.stride[1] == 1;
}
// [N*H*W, C] view of an image stored pixel by pixel, undefined for any other order in memory
Tensor pixel_rows(const Tensor& x) {
  const int64_t c = x.size(1), h = x.size(2), w = x.size(3);
  const bool pixels = x.stride(1) == 1 && x.stride(3) == c && x.stride(2) == w * c && x.stride(0) == h * w * c;
  return pixels ? x.as_strided({x.size(0) * h * w, c}, {c, 1}) : Tensor();
}

// [N*H*W, C] rows of a tensor stored plane by plane, in memory of their own
bool whole_planes(const Tensor& t) {
  return t.stride(3) == 1 && (t.size(2) == 1 || t.stride(2) == t.size(3)) && t.stride(1) >= t.size(2) * t.size(3) && t.size(1) > 1 &&
         t.size(2) * t.size(3) > 1;
}
Tensor rows_of_planes(const Tensor& t) {
  const int64_t pixels = t.size(2) * t.size(3);
  Tensor rows = new_matrix(t, t.size(0) * pixels, t.size(1));
  c10::DeviceGuard guard(t.device());
  check(sd_rows_from_planes(t.data_ptr(), t.stride(0), t.stride(1), rows.data_ptr(), t.size(0), t.size(1), pixels, stream_of(t)),
        "sd_rows_from_planes");
  return rows;
}
// The same of two tensors in one launch
std::pair<Tensor, Tensor> rows_of_planes(const Tensor& a, const Tensor& b) {
  Tensor out[2];
  const void* planes[2];
  void* rows[2];
  int64_t sn[2], sc[2], n[2], c[2], pixels[2];
  for (int i = 0; i < 2; ++i) {
    const Tensor& t = i ? b : a;
    n[i] = t.size(0);
    c[i] = t.size(1);
    pixels[i] = t.size(2) * t.size(3);
    out[i] = new_matrix(t, n[i] * pixels[i], c[i]);
    planes[i] = t.data_ptr();
    rows[i] = out[i].data_ptr();
    sn[i] = t.stride(0);
    sc[i] = t.stride(1);
  }
  c10::DeviceGuard guard(a.device());
  check(sd_conv2d_taps_prepare(2, planes, sn, sc, rows, n, c, pixels, nullptr, 0, 0, 0, 1, 1, 0, nullptr, nullptr, 0, 0, nullptr, 0, 0, 0.f,
                               dtype_of(a), stream_of(a)),
        "sd_conv2d_taps_prepare");
  return {out[0], out[1]};
}
// Whether that is the cheapest patch matrix of a pointwise kernel (own_patches)
bool turned(const Tensor& x, const ConvGeom& g) {
  return pointwise(g) && g.n > 0 && whole_planes(x) && g.rows() * g.c * 2 <= 64LL << 20;
}

// Which products of a masked convolution that the library takes without a patch matrix go through one all the same (the image is
// what is kept then too, and gathered once more for the kernel's gradient).  Measured on 298 drawn layers of 24 to 950 thousand
// rows; times through the matrix against those without, geometric means:
//  * forward: a workgroup takes 256 rows x 128 outputs and builds its tiles step by step; fewer than 64 of them 0.67 (9 x 96 x 8 x 8 ->
//    192, 5 x 5, p = 0.5, six of them: 45 us a pass for 306), 64 to 128 1.02, more 1.3; pointwise kernels, a step each, 1.04 to 1.3
//    gathered
//  * kernel's gradient: below 8192 rows 0.73, up to 16384 1.02, more 1.3; pointwise 0.90 below 16384 rows, above 1.16 gathered
//  * both of pointwise kernels whose image's planes are turned: passes of 14 layers that the GPU bounds 0.92 of those without, 1.00 at
//    worst (32 x 40 x 64 x 64 -> 176, p = 0.5 105 -> 85 us, 215 x 32 x 64 x 64 -> 56, p = 0.6 264 -> 222)
//  * input gradient, SDD and col2im against the fused kernel, both alone, 800 drawn geometries with kernels of 1 to 7 x 7, dilations and
//    strides of 1 to 4: 0.25 where the fold stages windows (344, nine of them above 1.05, 3 x 3 but for one, 1.46 at worst), but 0.59 with
//    the tile kernel (144, 33 above 1.1, 5.3 at worst: 128 x 32 x 32 x 32 -> 64, 3 x 3 by two down and one across, 83 -> 127 us a pass),
//    so the fused kernel keeps those.  Element by element 0.34 (311), 1.06 at worst but for unit strides with 64 outputs, where the fused
//    kernel's reduction is short and the fold's sums are not: of more than 8 million terms three in seven took longer, 1.7 at worst
//    (145 x 10 x 17 x 33 -> 64, 4 x 4, p = 0.25 112 -> 156 us a pass), of fewer 0.73 at worst.  1.03 to 1.09 where the matrix is one block
//    wide.  Past 256 MB it stays out of memory.
// Drawn from the generator's state the gather waits for a launch that draws (but for planes that are turned): passes of 180 layers of 4 to
// 256 images, kernels of 1 to 5 x 5, 0.61 of those without where the same seeds take 0.57, 1.001 at worst.  The matrices of rows this few
// stay under 0.9 GB (63 x 512 x 16 x 16 -> 64, 7 x 7, 809 MB, p = 0.5: 1590 us a pass for 1910).
bool forward_by_patches(const Tensor& x, const ConvGeom& g) {
  return turned(x, g) || (g.r * g.s > 1 && ceil_div(g.rows(), 256) * ceil_div(g.k, 128) < 64);
}
bool dw_by_patches(const Tensor& x, const ConvGeom& g) { return turned(x, g) || g.rows() < (g.r * g.s > 1 ? 8192 : 16384); }
bool dx_fuses(const Tensor& dy2, const Tensor& w2, const ConvGeom& g) {
  return sd_conv2d_dx_taken(dy2.data_ptr(), dy2.stride(0), w2.data_ptr(), w2.stride(0), GEOM_X(g), g.k, g.r, g.s, GEOM_W(g));
}
bool dx_by_patches(const ConvGeom& g, bool channels_last, int64_t bs) {
  if (g.cols() <= 64 || g.rows() * g.cols() * 2 > 256LL << 20) return false;
  if (pointwise(g) && channels_last) return true;  // written in place
  const int64_t sc = channels_last ? 1 : g.h * g.w, sw = channels_last ? g.c : 1;
  const int fold = sd_col2im_kernel(g.cols(), sc, g.w * sw, sw, GEOM_X(g), g.r, g.s, GEOM_W(g), bs);
  if (fold == SD_FOLD_ELEMENTS && g.stride[0] == 1 && g.stride[1] == 1 && g.k <= 64) return g.n * g.h * g.w * g.cols() <= 8 << 20;
  return fold != SD_FOLD_TILE;
}

// The patch matrix of a pointwise kernel: the image itself where it is its own, up to 64 MB the rows of its planes, else undefined.  Turning
// whole planes costs less than gathering the kept blocks of them, where blocks, rows and columns are looked up, as long as the caches hold
// what is moved: 35 x 24 x 56 x 56 at p = 0.5 12.4 us gathered, 4.6 turned; 30 x 256 x 14 x 14 7.6 and 3.6; 53 x 144 x 64 x 64 (62 MB) at
// p = 0.3 34 and 27, at p = 0.75 26 and 27; 200 x 200 x 56 x 56 (251 MB) at p = 0.6 98 and 152.
Tensor own_patches(const Tensor& x, const ConvGeom& g) {
  if (!pointwise(g) || g.n == 0) return Tensor();
  const Tensor own = g.c % 8 == 0 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 ? pixel_rows(x) : Tensor();
  return own.defined() || !turned(x, g) ? own : rows_of_planes(x);
}
Tensor im2col(const Tensor& x, const ConvGeom& g, const Lists* l) {
  const Tensor rows = own_patches(x, g);
  if (rows.defined()) return rows;
  Tensor cols = new_matrix(x, g.rows(), g.cols());
  c10::DeviceGuard guard(x.device());
  check(sd_im2col(x.data_ptr(), STRIDES4(x), cols.data_ptr(), cols.stride(0), GEOM_X(g), g.r, g.s, GEOM_W(g),
                  l ? l->row_ptr() : nullptr, l ? l->col_idx() : nullptr, l ? l->kernel_bs : 0, dtype_of(x),
                  stream_of(x)),
        "sd_im2col");
  return cols;
}

// Forward of a masked convolution through its patch matrix in two launches where there were three: the gather asks the mask's source
// (a stored mask or a seed), the product makes the lists.  cols: the patch matrix.
// A draw from the generator's state is made by one launch and read from what that stored: between two launches that each make it another
// stream may move the state on, and the product would read blocks that were not gathered.  Turning planes asks for no mask, so
// the launch that turns them makes the draw (31 x 16 x 16 x 16 -> 80, p = 0.75: the kernels of a pass 33 us with a launch of its own, 31 so).
Tensor patches_forward(const Tensor& x, const Tensor& w2, const ConvGeom& g, int64_t bs, double p, Draw draw, Lists& l, Tensor* cols) {
  check_conv_mask(g, bs, p, draw, l);
  if (draw.mask) draw.mask = check_mask(*draw.mask, l.mb, l.kb, x);
  c10::DeviceGuard guard(x.device());
  if (uint64_t* st = draw.state_ptr()) {  // (turned(x, g): the caller's business)
    l.allocate(x, OptTensor());
    *cols = new_matrix(x, g.rows(), g.c);
    const void* planes = x.data_ptr();
    void* rows = cols->data_ptr();
    const int64_t sn = x.stride(0), sc = x.stride(1), pixels = g.h * g.w;
    check(sd_conv2d_taps_prepare(1, &planes, &sn, &sc, &rows, &g.n, &g.c, &pixels, nullptr, 0, g.c, g.k, 1, 1, 0, nullptr,
                                 l.drawn(), l.mb, l.kb, st, 0, 0, (float)p, dtype_of(x), stream_of(x)),
          "sd_conv2d_taps_prepare");
    return layer_forward(*cols, w2, bs, p, draw, SD_ACT_NONE, false, l, nullptr, true);
  }
  *cols = own_patches(x, g);
  if (!cols->defined()) {
    *cols = new_matrix(x, g.rows(), g.cols());
    const MaskArg m = draw.mask ? MaskArg(*draw.mask) : MaskArg();
    check(sd_im2col_masked(x.data_ptr(), STRIDES4(x), cols->data_ptr(), cols->stride(0), GEOM_X(g), g.r, g.s, GEOM_W(g), m.ptr, m.sr,
                           m.sc, draw.seed.value_or(0), 0, (float)p, bs, dtype_of(x), stream_of(x)),
          "sd_im2col_masked");
  }
  return layer_forward(*cols, w2, bs, p, draw, SD_ACT_NONE, false, l, nullptr);
}
// Whether a layer's products take its operands as they are (else the calls one by one, which take any)
bool layer_takes(const ConvGeom& g, const Tensor& w2) { return g.cols() % 8 == 0 && g.k % 8 == 0 && rows_on_16_bytes(w2); }

Tensor conv_dw(const Tensor& x, const Tensor& dy2, const ConvGeom& g, const Lists* l, float scale) {
  Tensor dw = new_matrix(x, g.k, g.cols());
  Scratch ws(x, sd_conv2d_dw_workspace_bytes(g.n, g.c, g.k, g.r, g.s, g.po, g.qo));
  c10::DeviceGuard guard(x.device());
  const int rc = sd_conv2d_dw_lists(x.data_ptr(), STRIDES4(x), dy2.data_ptr(), dy2.stride(0), dw.data_ptr(),
                                    dw.stride(0), GEOM_X(g), g.k, g.r, g.s, GEOM_W(g), l ? l->col_ptr() : nullptr,
                                    l ? l->row_idx() : nullptr, l ? l->kernel_bs : 0, scale, dtype_of(x), ws.ptr,
                                    ws.bytes, stream_of(x));
  if (rc == SD_ERR_UNSUPPORTED) return Tensor();  // geometry not taken: nothing was launched
  check(rc, "sd_conv2d_dw_lists");
  return dw;
}

Tensor new_image(const Tensor& like, const ConvGeom& g, bool channels_last) {
  return at::empty({g.n, g.c, g.h, g.w}, like.options().memory_format(channels_last ? at::MemoryFormat::ChannelsLast
                                                                                     : at::MemoryFormat::Contiguous));
}

Tensor conv_dx(const Tensor& dy2, const Tensor& w2, const ConvGeom& g, const Lists* l, float scale, bool channels_last) {
  const MaskArg m = l ? l->mask() : MaskArg();
  Tensor dx = new_image(dy2, g, channels_last);
  c10::DeviceGuard guard(dy2.device());
  const int rc = sd_conv2d_dx_blocks(dy2.data_ptr(), dy2.stride(0), w2.data_ptr(), w2.stride(0), dx.data_ptr(), STRIDES4(dx),
                                     m.ptr, m.sr, m.sc, GEOM_X(g), g.k, g.r, g.s, GEOM_W(g), l ? l->bs : 64, scale, dtype_of(dy2),
                                     stream_of(dy2));
  if (rc == SD_ERR_UNSUPPORTED) return Tensor();
  check(rc, "sd_conv2d_dx_blocks");
  return dx;
}

// (N, K, P, Q) gradient -> [N*P*Q, K] row-major (free when it is channels-last in memory)
Tensor rows_gradient(const Tensor& grad, const ConvGeom& g, const Tensor& like) {
  Tensor d = grad.scalar_type() == like.scalar_type() ? grad : grad.to(like.scalar_type());
  if (whole_planes(d)) return rows_of_planes(d);
  d = d.permute({0, 2, 3, 1}).reshape({g.rows(), g.k});
  if (d.stride(1) != 1 || d.stride(0) < g.k) d = d.contiguous();  // e.g. the expanded (stride 0) gradient of a sum()
  return d;
}

// ---- the convolution tap by tap: images and gradients as rows of channels --------------------------------------------------
bool on_16_bytes(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// [N*H*W, C] view of an image whose pixels lie at one distance, as the tap-wise products read them, else undefined
Tensor pitched_rows(const Tensor& t) {
  const int64_t n = t.size(0), c = t.size(1), h = t.size(2), w = t.size(3);
  const int64_t ld = w > 1 ? t.stride(3) : (h > 1 ? t.stride(2) : (n > 1 ? t.stride(0) : c));
  const bool rows = t.stride(1) == 1 && ld >= c && ld % 8 == 0 && ld < (1 << 20) && (h == 1 || t.stride(2) == w * ld) &&
                    (n == 1 || t.stride(0) == h * w * ld) && on_16_bytes(t);
  return rows ? t.as_strided({n * h * w, c}, {ld, 1}) : Tensor();
}

// What one direction of it needs, in one launch: planes as rows, the packed weights, the mask.
struct TapsPrepare {
  int n = 0;
  const void* planes[2];
  void* rows[2];
  int64_t sn[2], sc[2], images[2], channels[2], pixels[2];
  std::vector<Tensor> keep;
  // t [N, C, H, W] as rows [N*H*W, C]: its own memory where its pixels lie at one distance, else a copy, from planes by the launch
  // (other slices of channels-last tensors are copied once, as they lie: by planes, in two passes, 128 x 64 x 32 x 32 -> 128
  // with a channel slice as the gradient took 207 us a pass, 184 before it went tap by tap)
  Tensor add(const Tensor& t_) {
    Tensor own = pitched_rows(t_);
    if (!own.defined() && t_.stride(1) == 1) own = pitched_rows(t_.contiguous(at::MemoryFormat::ChannelsLast));
    if (own.defined()) return own;
    Tensor t = t_;
    const int64_t h = t.size(2), w = t.size(3);
    const bool planar = (w == 1 || t.stride(3) == 1) && (h == 1 || t.stride(2) == w) && t.stride(1) >= h * w && t.stride(0) >= 1;
    if (!planar) t = t.contiguous();
    keep.push_back(t);
    Tensor out = new_matrix(t, t.size(0) * h * w, t.size(1));
    planes[n] = t.data_ptr();
    rows[n] = out.data_ptr();
    sn[n] = t.stride(0);
    sc[n] = t.stride(1);
    images[n] = t.size(0);
    channels[n] = t.size(1);
    pixels[n] = h * w;
    ++n;
    return out;
  }
  // w: the kernel as [K, C*R*S], undefined for none; draw: a mask for `lists`, or none
  Tensor launch(const Tensor& like, const Tensor& w, const ConvGeom& g, bool backward, double p, const Draw* draw, const Lists* lists) {
    Tensor packed;
    if (w.defined())
      packed = at::empty({sd_conv2d_taps_packed_bytes(g.c, g.k, g.r, g.s, backward) / 2}, like.options());
    const bool drawn = draw && !draw->mask;
    c10::DeviceGuard guard(like.device());
    check(sd_conv2d_taps_prepare(n, planes, sn, sc, rows, images, channels, pixels, w.defined() ? w.data_ptr() : nullptr, g.cols(),
                                 g.c, g.k, g.r, g.s, backward, packed.defined() ? packed.data_ptr() : nullptr,
                                 drawn ? lists->drawn() : nullptr, drawn ? lists->mb : 0, drawn ? lists->kb : 0,
                                 drawn ? draw->state_ptr() : nullptr, drawn ? draw->seed.value_or(0) : 0, 0, (float)p,
                                 dtype_of(like), stream_of(like)),
          "sd_conv2d_taps_prepare");
    return packed;
  }
};
#define MASK_OF(m, l) (m).ptr, (m).sr, (m).sc, (l) ? (l)->bs : 0

Tensor taps_forward(const Tensor& rows, const Tensor& packed, const ConvGeom& g, const Lists* l, float scale) {
  Tensor y2 = new_matrix(rows, g.rows(), g.k);
  const MaskArg m = l ? l->mask() : MaskArg();
  c10::DeviceGuard guard(rows.device());
  check(sd_conv2d_taps_forward(rows.data_ptr(), rows.stride(0), packed.data_ptr(), y2.data_ptr(), g.k, MASK_OF(m, l), GEOM_X(g), g.k,
                               g.r, g.s, GEOM_W(g), scale, dtype_of(rows), stream_of(rows)),
        "sd_conv2d_taps_forward");
  return y2;
}

struct ConvBackward : Node {
  // the kernel as [K, C*R*S], and what the kernel's gradient reads or is gathered from: the image in the geometries that the
  // implicit products take, whichever way the forward went, and where a pointwise kernel's patch matrix is the image's own pixels,
  // else the patch matrix that the forward made
  // (tap by tap: the image's rows when the forward made a copy of them that nothing else refers to, else the image)
  Saved w2, x, cols;
  SavedLists saved;  // nothing kept: no dropout
  ConvGeom g{};
  double p = 0;
  bool fused_dx = true, channels_last = false, pixels = false, taps = false;
  // tap by tap: `w` the kernel as a matrix, `image` or `kept_rows` whichever was kept
  variable_list apply_taps(const Tensor& grad, const Tensor& w, const Tensor& image, Tensor rows, const Lists* l) {
    variable_list out(2);
    const bool need_dx = task_should_compute_output(0), need_dw = task_should_compute_output(1);
    const float scale = (float)(1.0 / (1.0 - p));
    TapsPrepare prepare;
    Tensor d = grad.defined() ? grad : at::zeros({g.n, g.k, g.po, g.qo}, w.options());
    if (d.scalar_type() != w.scalar_type()) d = d.to(w.scalar_type());
    const Tensor dy2 = prepare.add(d);
    if (rows.defined()) {
      if (rows.stride(1) != 1 || rows.stride(0) != g.c || !on_16_bytes(rows)) rows = rows.clone(at::MemoryFormat::Contiguous);
    } else if (need_dw) {
      rows = prepare.add(image);
    }
    const Tensor packed = prepare.launch(d, need_dx ? w : Tensor(), g, true, 0.0, nullptr, nullptr);
    const MaskArg m = l ? l->mask() : MaskArg();
    c10::DeviceGuard guard(d.device());
    if (need_dx) {
      Tensor dx = new_image(dy2, g, channels_last);
      check(sd_conv2d_taps_dx(dy2.data_ptr(), dy2.stride(0), packed.data_ptr(), dx.data_ptr(), STRIDES4(dx), MASK_OF(m, l), GEOM_X(g),
                              g.k, g.r, g.s, GEOM_W(g), scale, dtype_of(d), stream_of(d)),
            "sd_conv2d_taps_dx");
      last_routes[1] = kFused;
      out[0] = dx;
    }
    if (need_dw) {
      Tensor dw = new_matrix(dy2, g.k, g.cols());
      Scratch ws(d, sd_conv2d_taps_dw_workspace_bytes(g.c, g.k, g.r, g.s, g.rows()));
      check(sd_conv2d_taps_dw(rows.data_ptr(), rows.stride(0), dy2.data_ptr(), dy2.stride(0), dw.data_ptr(), dw.stride(0),
                              MASK_OF(m, l), GEOM_X(g), g.k, g.r, g.s, GEOM_W(g), scale, dtype_of(d), ws.ptr, ws.bytes, stream_of(d)),
            "sd_conv2d_taps_dw");
      last_routes[2] = kImplicit;
      out[1] = dw.view({g.k, g.c, g.r, g.s});
    }
    return out;
  }
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    at::NoGradGuard no_grad;
    variable_list out(2);
    const Tensor w = w2.get().contiguous(), image = x.get();
    const Lists lists = saved.get();
    Tensor patches = cols.matrix();
    if (taps) return apply_taps(grads[0], w, image, patches, lists.buf.defined() ? &lists : nullptr);
    const Lists* l = lists.buf.defined() ? &lists : nullptr;
    const float scale = (float)(1.0 / (1.0 - p));
    Tensor dy2;
    // the image of a pointwise kernel is turned with the output gradient (31 x 16 x 16 x 16 -> 80, p = 0.75: the kernels of a pass 31 us
    // with a launch for either, 29 so; 60 x 64 x 64 x 64 -> 64, p = 0.1 148 and 143)
    if (l && task_should_compute_output(1) && !patches.defined() && grads[0].defined() && grads[0].scalar_type() == w.scalar_type() &&
        whole_planes(grads[0]) && turned(image, g))
      std::tie(dy2, patches) = rows_of_planes(grads[0], image);
    else
      dy2 = grads[0].defined() ? rows_gradient(grads[0], g, w) : at::zeros({g.rows(), g.k}, w.options());
    // both gradients through the patch matrix: one launch where the pair qualifies, and the fold
    const bool fused = fused_dx && !(l && dx_by_patches(g, channels_last, l->bs)) && dx_fuses(dy2, w, g);
    const bool dw_through = pixels || patches.defined() || dw_by_patches(image, g);
    if (l && task_should_compute_output(0) && task_should_compute_output(1) && dw_through && !fused && layer_takes(g, w) && rows_on_16_bytes(dy2)) {
      if (!patches.defined()) patches = im2col(image, g, l);
      if (rows_on_16_bytes(patches)) {
        // a pointwise kernel's patch gradient is that of a channels-last image: the product writes it in place, zeros included
        const bool in_place = pointwise(g) && channels_last;
        auto [dcols, dk] = layer_products(dy2, w, patches, *l, p, true, true, SD_ACT_NONE, Tensor(), !in_place);
        last_routes[1] = last_routes[2] = kExplicit;
        if (in_place) {
          out[0] = dcols.view({g.n, g.h, g.w, g.c}).permute({0, 3, 1, 2});
        } else {
          Tensor dx = new_image(dy2, g, channels_last);
          const MaskArg m = l->mask();
          c10::DeviceGuard guard(dy2.device());
          check(sd_col2im(dcols.data_ptr(), dcols.stride(0), dx.data_ptr(), STRIDES4(dx), GEOM_X(g), g.r, g.s, GEOM_W(g), m.ptr,
                          m.sr, m.sc, l->bs, dtype_of(dy2), stream_of(dy2)),
                "sd_col2im");
          out[0] = dx;
        }
        out[1] = dk.view({g.k, g.c, g.r, g.s});
        return out;
      }
    }
    if (task_should_compute_output(0)) {
      Tensor dx;
      if (fused) dx = conv_dx(dy2, w, g, l, scale, channels_last);
      last_routes[1] = dx.defined() ? kFused : kExplicit;
      if (!dx.defined()) {
        dx = new_image(dy2, g, channels_last);
        // a pointwise kernel's patch gradient is the image's: the product writes it in place, zeros included (238 x 96 x
        // 14 x 14 -> 168, p = 0.5, both directions: 118 us with the copies, 64 without)
        const Tensor in_place = pointwise(g) ? pixel_rows(dx) : Tensor();
        Tensor dcols = in_place.defined() ? in_place : new_matrix(dy2, g.rows(), g.cols());
        const Mat gm(dy2), dm(dcols);
        const Mat wt(w.t());
        c10::DeviceGuard guard(dy2.device());
        MaskArg m;
        if (l) {
          // col2im skips the dropped blocks, so the product need not zero them
          check(sd_gemm_sdd_lists_ex(MAT(gm), MAT(wt), MAT(dm), l->row_ptr(), l->col_idx(), g.rows(), g.cols(), g.k,
                                     l->kernel_bs, scale, dtype_of(dy2), in_place.defined() ? 0 : 1, 1.f / scale, stream_of(dy2)),
                "sd_gemm_sdd_lists_ex");
          m = l->mask();
        } else {
          Scratch ws(dy2, sd_splitk_workspace_bytes(g.rows(), g.cols(), g.k, 0, 0));
          check(sd_gemm(MAT(gm), MAT(wt), MAT(dm), g.rows(), g.cols(), g.k, dtype_of(dy2), ws.ptr, ws.bytes,
                        stream_of(dy2)),
                "sd_gemm");
        }
        if (!in_place.defined())
          check(sd_col2im(dcols.data_ptr(), dcols.stride(0), dx.data_ptr(), STRIDES4(dx), GEOM_X(g), g.r, g.s,
                          GEOM_W(g), m.ptr, m.sr, m.sc, l ? l->bs : 0, dtype_of(dy2), stream_of(dy2)),
                "sd_col2im");
      }
      out[0] = dx;
    }
    if (task_should_compute_output(1)) {
      Tensor dk;
      if (pixels) patches = im2col(image, g, l);
      if (!patches.defined()) {  // the image was kept
        if (!(l && dw_by_patches(image, g))) dk = conv_dw(image, dy2, g, l, scale);
        if (!dk.defined()) patches = im2col(image, g, l);
      }
      last_routes[2] = dk.defined() ? kImplicit : kExplicit;
      if (!dk.defined()) {
        dk = new_matrix(dy2, g.k, g.cols());
        const Mat am(patches.t()), bm(dy2.t()), cm(dk.t());
        c10::DeviceGuard guard(dy2.device());
        if (l) {
          Scratch ws(dy2, sd_splitk_workspace_bytes(g.cols(), g.k, g.rows(), l->kernel_bs, 1));
          check(sd_gemm_dsd_lists(MAT(am), MAT(bm), MAT(cm), l->col_ptr(), l->row_idx(), g.cols(), g.k, g.rows(),
                                  l->kernel_bs, scale, dtype_of(dy2), ws.ptr, ws.bytes, stream_of(dy2)),
                "sd_gemm_dsd_lists");
        } else {
          Scratch ws(dy2, sd_splitk_workspace_bytes(g.cols(), g.k, g.rows(), 0, 0));
          check(sd_gemm(MAT(am), MAT(bm), MAT(cm), g.cols(), g.k, g.rows(), dtype_of(dy2), ws.ptr, ws.bytes,
                        stream_of(dy2)),
                "sd_gemm");
        }
      }
      out[1] = dk.view({g.k, g.c, g.r, g.s});
    }
    return out;
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (Saved* s : {&x, &w2, &cols}) s->drop();
    saved.drop();
  }
  std::string name() const override { return "Im2colConv2dBackward"; }
};

using Pair = std::array<int64_t, 2>;

// block size 0: no dropout
Tensor conv2d(const Tensor& input, const Tensor& kernel_in, const OptTensor& mask, int64_t bs, double p,
              const Pair& padding, const Pair& stride, const Pair& dilation, std::optional<uint64_t> seed,
              const OptTensor& state, bool implicit_forward, bool fused_dx) {
  TORCH_CHECK_VALUE(input.dim() == 4 && kernel_in.dim() == 4, "input must be (N, C, H, W) and kernel (K, C, R, S)");
  TORCH_CHECK_VALUE(input.size(1) == kernel_in.size(1), "channel mismatch: input ", input.size(1), ", kernel ",
                    kernel_in.size(1));
  for (int i = 0; i < 2; ++i)  // (before anything is divided by them)
    TORCH_CHECK_VALUE(stride[i] > 0 && dilation[i] > 0 && padding[i] >= 0,
                      "strides and dilations must be positive, paddings non-negative");
  const Tensor x = autocast(input), kernel = autocast(kernel_in).contiguous();
  refuse_forward_mode(std::array<Tensor, 2>{x, kernel});
  TORCH_CHECK_VALUE(x.is_cuda() && (x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16),
                    "x must be a 4D float16/bfloat16 tensor on the GPU");
  TORCH_CHECK_VALUE(kernel.scalar_type() == x.scalar_type() && kernel.device() == x.device(), "kernel must be a ",
                    x.dtype(), " tensor on ", x.device());
  ConvGeom g{x.size(0), x.size(1), x.size(2), x.size(3), kernel.size(0), kernel.size(2), kernel.size(3)};
  for (int i = 0; i < 2; ++i) {
    g.pad[i] = padding[i];
    g.stride[i] = stride[i];
    g.dil[i] = dilation[i];
  }
  auto out_size = [](int64_t in, int64_t pad, int64_t dil, int64_t taps, int64_t step) {
    const int64_t room = in + 2 * pad - dil * (taps - 1) - 1;
    return room < 0 ? 0 : room / step + 1;
  };
  g.po = out_size(g.h, g.pad[0], g.dil[0], g.r, g.stride[0]);
  g.qo = out_size(g.w, g.pad[1], g.dil[1], g.s, g.stride[1]);
  TORCH_CHECK_VALUE(g.po > 0 && g.qo > 0, "kernel does not fit the padded image");
  TORCH_CHECK_VALUE(g.k > 0 || !implicit_forward, "the kernel has no outputs");  // (the implicit products' refusal, on every route)
  Lists lists;
  Tensor y, y2, cols;
  const float scale = bs ? (float)(1.0 / (1.0 - p)) : 1.f;
  const bool taps = implicit_forward && fused_dx && sd_conv2d_taps_taken_blocks(GEOM_X(g), g.k, g.r, g.s, GEOM_W(g), bs ? p : 0.0, bs);
  const bool record = records(std::array<Tensor, 2>{x, kernel});
  bool keeps_input = true;
  if (taps) {
    NoRecord guard;
    lists.mask_only = true;
    const Draw draw{mask, seed, state};
    if (bs) conv_mask(x, g, bs, p, draw, lists);
    const Lists* l = bs ? &lists : nullptr;
    TapsPrepare prepare;
    Tensor rows = prepare.add(x);
    const Tensor packed = prepare.launch(x, kernel, g, false, p, l ? &draw : nullptr, l);
    y2 = taps_forward(rows, packed, g, l, scale);
    last_routes[0] = kImplicit;
    last_routes[1] = last_routes[2] = kNone;
    // What is kept for the kernel's gradient, the image or its rows, follows what the other routes keep, the image or its
    // patch matrix: a write to the image before the backward is refused or allowed in the same geometries.
    const bool keeps_image = sd_conv2d_implicit_taken(x.data_ptr(), STRIDES4(x), kernel.data_ptr(), g.cols(), GEOM_X(g), g.k, g.r, g.s, GEOM_W(g));
    // (Without a gradient for the kernel the rows are not read again, and not kept: a clone of 26 MB at 128 x 128 x 28 x 28.)
    keeps_input = keeps_image;
    if (record && !keeps_image && kernel.requires_grad()) cols = rows.is_alias_of(x) ? rows.clone() : rows;
    y = y2.view({g.n, g.po, g.qo, g.k}).permute({0, 3, 1, 2});
  } else {
    NoRecord guard;
    const Lists* l = bs ? &lists : nullptr;
    bool done = false;
    c10::DeviceGuard device(x.device());
    const Tensor w2 = kernel.detach().view({g.k, g.cols()});  // (not what is kept: below autograd it has no part in kernel's version)
    const bool takes_implicit = implicit_forward && sd_conv2d_implicit_taken(x.data_ptr(), STRIDES4(x), kernel.data_ptr(), g.cols(),
                                                                              GEOM_X(g), g.k, g.r, g.s, GEOM_W(g));
    const Draw draw{mask, seed, state};
    const bool implicit = takes_implicit && !(bs && forward_by_patches(x, g));
    const bool layer = bs && layer_takes(g, w2) && (!draw.state_ptr() || turned(x, g));  // (see patches_forward)
    if (implicit || !layer) {
      if (bs) conv_lists(x, g, bs, p, draw, lists);
      y2 = new_matrix(x, g.rows(), g.k);
    }
    if (implicit) {  // no patch matrix in memory
      const int rc = sd_conv2d_dsd_lists(x.data_ptr(), STRIDES4(x), kernel.data_ptr(), g.cols(), y2.data_ptr(),
                                         y2.stride(0), GEOM_X(g), g.k, g.r, g.s, GEOM_W(g), l ? l->row_ptr() : nullptr,
                                         l ? l->col_idx() : nullptr, l ? l->kernel_bs : 0, scale, dtype_of(x),
                                         stream_of(x));
      if (rc != SD_ERR_UNSUPPORTED) check(rc, "sd_conv2d_dsd_lists");
      done = rc == SD_OK;
    }
    last_routes[0] = done ? kImplicit : kExplicit;
    last_routes[1] = last_routes[2] = kNone;
    if (!done && layer && !implicit) {
      y2 = patches_forward(x, w2, g, bs, p, draw, lists, &cols);
    } else if (!done) {
      cols = im2col(x, g, l);
      Mat am(cols), bm, cm(y2);
      bm.ptr = kernel.data_ptr();
      bm.sr = std::max<int64_t>(g.cols(), 1);
      bm.sc = 1;
      Scratch ws(x, sd_splitk_workspace_bytes(g.rows(), g.k, g.cols(), l ? l->kernel_bs : 0, l ? 1 : 0));
      if (l)
        check(sd_gemm_dsd_lists(MAT(am), MAT(bm), MAT(cm), l->row_ptr(), l->col_idx(), g.rows(), g.k, g.cols(),
                                l->kernel_bs, scale, dtype_of(x), ws.ptr, ws.bytes, stream_of(x)),
              "sd_gemm_dsd_lists");
      else
        check(sd_gemm(MAT(am), MAT(bm), MAT(cm), g.rows(), g.k, g.cols(), dtype_of(x), ws.ptr, ws.bytes, stream_of(x)),
              "sd_gemm");
    }
    // (in the geometries that the implicit products take the image is kept, and gathered once more for the kernel's gradient)
    if (takes_implicit) cols = Tensor();
    // the result is an (N, K, P, Q) view of an (N, P*Q, K) buffer, as the reference's is (im2col_conv2d.py:26-27)
    y = y2.view({g.n, g.po, g.qo, g.k}).permute({0, 3, 1, 2});
  }
  if (record) {
    auto node = make_node<ConvBackward>({x, kernel});
    node->taps = taps;
    node->pixels = cols.defined() && cols.is_alias_of(x);
    if (cols.defined() && !node->pixels) node->cols.keep(cols);
    else if (keeps_input) node->x.keep(x);
    node->w2.keep(kernel.detach().view({g.k, g.cols()}));
    if (bs) node->saved.keep(std::move(lists), mask.value_or(Tensor()));
    node->g = g;
    node->p = bs ? p : 0.0;
    node->fused_dx = fused_dx;
    node->channels_last = x.is_contiguous(at::MemoryFormat::ChannelsLast) && !x.is_contiguous();
    torch::autograd::set_history(y, node);
  }
  return y;
}

std::array<int, 3> conv_routes() { return {last_routes[0].load(), last_routes[1].load(), last_routes[2].load()}; }

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  namespace py = pybind11;
  m.def("source_hash", [] { return SD_SOURCE_HASH; });
  m.def("set_library_error", [](py::object cls) { library_error = cls.release().ptr(); });
  m.def("linear", torch::wrap_pybind_function(linear));
  m.def("mlp", torch::wrap_pybind_function(mlp));
  m.def("conv2d", torch::wrap_pybind_function(conv2d));
  m.def("conv_routes", &conv_routes);
}
