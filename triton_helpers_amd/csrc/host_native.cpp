// The host side of the operators in native code: argument checks, allocation, the call into libnf_cdna4.so and the autograd
// nodes.  What a small call costs is the host: as Python functions under torch.autograd.Function a forward + backward of the
// fused MLP at 64 rows took 66 us of interpreter, ctypes and engine time around 25 us of kernels, with the backward waiting
// for the interpreter lock on the engine's thread.
//
// Each operator's function here takes the plain case (GPU tensors, no tracing, tangents or other modes) and returns None for everything
// else, an argument error included: the Python function of the operator then takes over, which holds the full checks and
// their messages.  Both come to the same launch functions below.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <array>
#include <cstring>
#include <memory>
#include <mutex>
#include <optional>
#include <vector>

#include "nf_cdna4.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ------------------------------------------------------------------------------------------------ pieces
int code_of(at::ScalarType t) {
  return t == at::kFloat ? NF_F32 : t == at::kHalf ? NF_F16 : t == at::kBFloat16 ? NF_BF16 : -1;
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

Tensor contiguous(const Tensor& t) { return t.defined() && !t.is_contiguous() ? t.contiguous() : t; }

void check(int rc, const char* what) { TORCH_CHECK(rc == 0, what, " failed (code ", rc, "): ", nf_last_error()); }

Tensor scratch(int64_t bytes, const Tensor& like) {
  return bytes > 0 ? at::empty({bytes}, like.options().dtype(at::kByte)) : Tensor();
}

// A tensor as rows of `width`: address, row stride and count.  Rows that overlap (an expanded tensor has row stride 0) or a
// strided inner dimension are copied.
struct Rows {
  Tensor hold;
  void* p;
  int64_t n, stride;
  Rows(const Tensor& t, int64_t width) : hold(t), n(t.numel() / width), stride(width) {
    if (!t.is_contiguous()) {
      hold = t.reshape({-1, width});
      if (hold.stride(1) != 1 || (n > 1 && hold.stride(0) < width)) hold = hold.contiguous();
      stride = hold.stride(0);
    }
    p = hold.data_ptr();
  }
};

// One buffer for the gradients of several parameters, in pieces on 16-byte boundaries.
struct Pieces {
  std::array<int64_t, 6> offset{};
  int64_t total = 0;
  template <size_t K>
  Pieces(const std::array<Tensor, K>& like, int64_t unit) {
    for (size_t i = 0; i < K; ++i) {
      offset[i] = total;
      if (like[i].defined()) total += (like[i].numel() + unit - 1) / unit * unit;
    }
  }
  void* at(const Tensor& flat, const Tensor& like, int i) const {
    return like.defined() ? (char*)flat.data_ptr() + offset[i] * flat.element_size() : nullptr;
  }
  Tensor view(const Tensor& flat, const Tensor& like, int i) const {
    return like.defined() ? flat.as_strided(like.sizes(), like.strides(), flat.storage_offset() + offset[i]) : Tensor();
  }
};

// ------------------------------------------------------------------------------------------------ hash encoding
struct Geometry {
  std::array<int64_t, 6> key;  // T, levels, D, F, min_res, max_res
  nf_hash_geom g;
  int64_t rows;
};

// Filled from Python, where the level arithmetic lives; entries stay for the life of the process (nodes point at them).
constexpr size_t MAX_GEOMETRIES = 1024;
std::vector<std::unique_ptr<Geometry>>& geometries() {
  static auto* v = new std::vector<std::unique_ptr<Geometry>>();
  return *v;
}

const Geometry* find_geometry(const std::array<int64_t, 6>& key) {  // under the interpreter lock
  static const Geometry* last = nullptr;
  if (last != nullptr && last->key == key) return last;
  for (auto& e : geometries())
    if (e->key == key) return last = e.get();
  return nullptr;
}

// The paper's primes on a GPU, made once per process for all callers, the Python functions among them: as an ordinary tensor, whatever
// the mode of the first call (an inference tensor could not be saved for a backward later, a wrapper of a mode would outlive it).
Tensor default_primes(c10::Device device) {
  static std::mutex m;
  static auto* by_device = new std::vector<Tensor>();
  std::lock_guard<std::mutex> lock(m);
  const size_t i = device.index();
  if (by_device->size() <= i) by_device->resize(i + 1);
  Tensor& t = (*by_device)[i];
  if (!t.defined()) {
    const c10::DeviceGuard guard(device);
    TORCH_CHECK(c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None,
                "the first call of the hash encoding on a device copies its primes there: make one before capturing a graph");
    const c10::InferenceMode ordinary(false);
    using K = c10::DispatchKey;
    const c10::impl::ExcludeDispatchKeyGuard no_modes(c10::DispatchKeySet(
        {K::Python, K::PythonTLSSnapshot, K::Functionalize, K::FuncTorchVmapMode, K::FuncTorchDynamicLayerFrontMode, K::FuncTorchDynamicLayerBackMode, K::Tracer}));
    t = at::tensor(at::ArrayRef<int64_t>({1, 2654435761ll, 805459861ll}), at::kLong).to(device);
  }
  return t;
}

constexpr int64_t REPACK_MIN_POINTS = 4096;  // gradient rows off 16-byte boundaries are packed first from this many on

Tensor encode_forward(const Tensor& coords, const Tensor& table, const Tensor& pi, const Geometry& geo, double scale, int64_t flags) {
  const c10::DeviceGuard guard(coords.device());
  const int64_t D = coords.size(-1), width = geo.g.levels * geo.g.feat;
  c10::SmallVector<int64_t, 5> shape(coords.sizes().begin(), coords.sizes().end());
  shape.back() = width;
  Tensor out = at::empty(shape, table.options());
  const Tensor c = coords.is_contiguous() ? coords : coords.reshape({-1, D});
  const bool flat = coords.is_contiguous();
  check(nf_hash_encode_fwd(c.data_ptr(), code_of(c.scalar_type()), flat ? D : c.stride(0), flat ? 1 : c.stride(1), table.data_ptr(),
                           code_of(table.scalar_type()), out.data_ptr(), width, out.numel() / width, &geo.g, pi.data_ptr<int64_t>(),
                           (float)scale, (int)flags, stream_of(coords)),
        "nf_hash_encode_fwd");
  return out;
}

// The upstream gradient as rows that the kernels take, the scratch, and the point coordinates of a backward.
struct BackwardArgs {
  Rows rows;
  Tensor c, ws;
  int64_t n, csn, csd, bytes;
  int dt;
  BackwardArgs(const Tensor& coords, const Tensor& grad, const nf_hash_geom& g, int64_t flags) : rows(grad, grad.size(-1)) {
    const int64_t D = coords.size(-1);
    n = coords.numel() / D;
    if (rows.n >= REPACK_MIN_POINTS && (rows.stride * grad.element_size() % 16 != 0 || (uintptr_t)rows.p % 16 != 0)) {
      // gradient rows off 16-byte boundaries (the output carried appended features): the LDS-tile kernels read whole aligned
      // rows, so the encoding's columns are packed first (one pass instead of scattered atomics per corner)
      const int64_t width = g.levels * g.feat;
      rows.hold = rows.hold.reshape({-1, grad.size(-1)}).narrow(1, 0, width).clone(at::MemoryFormat::Contiguous);
      rows.p = rows.hold.data_ptr();
      rows.stride = width;
    }
    dt = code_of(grad.scalar_type());
    const bool flat = coords.is_contiguous();
    c = flat ? coords : coords.reshape({-1, D});
    csn = flat ? D : c.stride(0);
    csd = flat ? 1 : c.stride(1);
    bytes = nf_hash_encode_bwd_workspace_bytes(n, &g, dt, (int)flags);
    ws = scratch(bytes, coords);
  }
};

void encode_backward_add(const BackwardArgs& a, const Tensor& de, const Tensor& pi, const nf_hash_geom& g, double scale, int64_t flags) {
  check(nf_hash_encode_bwd(a.c.data_ptr(), code_of(a.c.scalar_type()), a.csn, a.csd, a.rows.p, a.dt, a.rows.stride, de.data_ptr<float>(), a.n, &g,
                           pi.data_ptr<int64_t>(), (float)scale, ptr(a.ws), a.bytes, (int)flags, stream_of(a.c)),
        "nf_hash_encode_bwd");
}

// adds into de
void encode_backward(const Tensor& coords, const Tensor& grad, const Tensor& de, const Tensor& pi, const nf_hash_geom& g, double scale, int64_t flags) {
  const c10::DeviceGuard guard(coords.device());
  encode_backward_add(BackwardArgs(coords, grad, g, flags), de, pi, g, scale, flags);
}

// the gradient of `table`: in its own type where the kernels write it whole, else float32 sums that autograd rounds to that type
Tensor encode_table_grad(const Tensor& coords, const Tensor& grad, const Tensor& table, const Tensor& pi, const Geometry& geo, double scale, int64_t flags) {
  const c10::DeviceGuard guard(coords.device());
  const BackwardArgs a(coords, grad, geo.g, flags);
  if (table.size(0) == geo.rows && a.bytes > 0) {
    const Tensor de = at::empty(table.sizes(), table.options());
    const int rc = nf_hash_encode_bwd_write(a.c.data_ptr(), code_of(a.c.scalar_type()), a.csn, a.csd, a.rows.p, a.dt, a.rows.stride, de.data_ptr(),
                                            code_of(table.scalar_type()), a.n, &geo.g, pi.data_ptr<int64_t>(), (float)scale, ptr(a.ws), a.bytes,
                                            (int)flags, stream_of(a.c));
    if (rc != NF_EUNSUPPORTED) {
      check(rc, "nf_hash_encode_bwd_write");
      return de;
    }
  }
  const Tensor de = at::zeros(table.sizes(), table.options().dtype(at::kFloat));
  encode_backward_add(a, de, pi, geo.g, scale, flags);
  return de;
}

// In the nodes' backwards the saved tensors are unpacked first: that runs the user's saved-tensor hooks (checkpointing recomputes its
// region there), which need autograd on.
struct HashEncoding : torch::autograd::Function<HashEncoding> {
  static Tensor forward(AutogradContext* ctx, const Tensor& coords, const Tensor& table, const Tensor& pi, const Geometry* geo, double scale,
                        int64_t flags) {
    const at::AutoDispatchBelowADInplaceOrView below;
    ctx->save_for_backward({coords, table, pi});
    ctx->saved_data["geometry"] = (int64_t)(uintptr_t)geo;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["flags"] = flags;
    return encode_forward(coords, table, pi, *geo, scale, flags);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const at::AutoDispatchBelowADInplaceOrView below;
    const auto* geo = (const Geometry*)(uintptr_t)ctx->saved_data["geometry"].toInt();
    const Tensor de = encode_table_grad(saved[0], grads[0], saved[1], saved[2], *geo, ctx->saved_data["scale"].toDouble(), ctx->saved_data["flags"].toInt());
    return {Tensor(), de, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// ------------------------------------------------------------------------------------------------ fused MLP
struct Mlp {
  Tensor x;
  std::array<Tensor, 6> w;  // w_in, b_in, w_out, b_out, w_hid, b_hid
  int act = 0;
  int64_t depth() const { return w[4].defined() ? w[4].size(0) / w[0].size(0) + 1 : 1; }
  int64_t d_in() const { return w[0].size(1); }
  int64_t d_hidden() const { return w[0].size(0); }
  int64_t d_out() const { return w[2].size(0); }
};

Tensor mlp_forward(Mlp m) {
  const c10::DeviceGuard guard(m.x.device());
  for (Tensor& t : m.w) t = contiguous(t);
  const Rows x(m.x, m.d_in());
  Tensor y = at::empty({m.x.size(0), m.x.size(1), m.d_out()}, m.w[0].options());
  const int dt = code_of(m.w[0].scalar_type());
  const int64_t bytes = nf_mlp_workspace_bytes(x.n, (int)m.d_hidden(), (int)m.depth(), m.act, 0, dt);
  const Tensor ws = scratch(bytes, m.x);
  check(nf_mlp_fwd(x.p, x.stride, y.data_ptr(), m.d_out(), ptr(m.w[0]), ptr(m.w[1]), ptr(m.w[4]), ptr(m.w[5]), ptr(m.w[2]), ptr(m.w[3]), x.n,
                   (int)m.d_in(), (int)m.d_hidden(), (int)m.d_out(), (int)m.depth(), m.act, dt, code_of(m.x.scalar_type()), ptr(ws), bytes,
                   stream_of(m.x)),
        "nf_mlp_fwd");
  return y;
}

// (dx, dw_in, db_in, dw_out, db_out, dw_hid, db_hid); the parameters' gradients in their own dtype, or as float32
variable_list mlp_backward(Mlp m, Tensor dy, bool need_dx, bool float_grads) {
  const c10::DeviceGuard guard(m.x.device());
  for (Tensor& t : m.w) t = contiguous(t);
  const auto wt = m.w[0].scalar_type();
  const int dt = code_of(wt), H = (int)m.d_hidden(), in = (int)m.d_in(), out = (int)m.d_out(), depth = (int)m.depth();
  const bool relu = m.act == NF_ACT_RELU;
  if (dy.scalar_type() != wt) dy = dy.to(wt);
  const Rows g(dy, out);
  Rows x(m.x, in);
  // Up to nine hidden layers: one launch for the whole backward, but where the kernels that nf_mlp_bwd chains stream many rows faster than
  // its LDS does.  64 wide on whole 8-byte pieces, us whole / chained: 32 -> 16 with two layers of another activation than ReLU 2^19 rows 85 / 84, 0.8 M
  // 118 / 107, 2^20 142 / 132 (64 -> 64 197 / 272); with three ReLU layers 0.8 M 113 / 108, 1.5 M 187 / 167, 2^21 260 / 220 (64 -> 64 269 / 267 and
  // 367 / 355 at the last two); five 381 / 373 and 527 / 497 (64 -> 64 442 / 438 and 605 / 580).  Whole is faster or as fast with four (1.5 M 236 / 254),
  // six (433 / 448) and from seven on (563 / 585, nine 685 / 699; 64 -> 64 618 / 671, 739 / 763), in either type, and on other rows: 32 -> 16
  // off 8-byte boundaries 0.8 M 122 / 155, 35 -> 3 with three layers 1.5 M 244 / 364.
  const auto pieces = [](const Rows& r, int width) { return width % 4 == 0 && r.stride % 4 == 0 && (uintptr_t)r.p % 8 == 0; };
  const bool narrow = in <= 32 && out <= 16;
  const bool streams = H == 64 && m.x.scalar_type() == wt && pieces(x, in) && pieces(g, out) &&
                       (depth == 2 ? narrow && g.n > 3 << 18 : relu && (depth == 3 || depth == 5) && g.n > (narrow && depth == 3 ? 3 << 18 : 7 << 18));
  const int64_t whole_bytes = streams ? 0 : nf_mlp_bwd_whole_workspace_bytes(g.n, H, depth, m.act, dt);
  if (m.x.scalar_type() != wt && whole_bytes == 0) {  // deeper networks, no rows
    m.x = m.x.to(wt);
    x = Rows(m.x, in);
  }
  Tensor flat, dx;
  const auto finish = [&](const Pieces& at, const Tensor& f) {
    return variable_list{dx, at.view(f, m.w[0], 0), at.view(f, m.w[1], 1), at.view(f, m.w[2], 2), at.view(f, m.w[3], 3), at.view(f, m.w[4], 4),
                         at.view(f, m.w[5], 5)};
  };
  const bool decoder = in <= 32 && out <= 16;  // the wider shapes need x in the parameters' dtype
  // ReLU at 64 wide has kernels of its own for one and two hidden layers, which lay their weights out in both forms, sum eight waves
  // and (one hidden layer) go through an identity layer: quicker than the whole backward from about 2^16 rows, at one layer from 2^19 where
  // the output is narrow (us own / whole: 32 -> 64 -> 64 -> 16 2^12 rows 14.9 / 9.8, 2^16 19.4 / 18.6, 2^17 22 / 24, 2^20 60 / 102; 64 -> 64 -> 64
  // -> 64 2^16 22.2 / 22.3, 2^17 25.5 / 29.7; 32 -> 64 -> 16 2^18 27.8 / 25.1, 2^19 38.2 / 39.1, 2^20 61 / 70).  One layer with a wide output takes the whole
  // backward in every batch: it is the quicker one of narrow inputs and below 2^19 rows (2^20 rows 16 -> 64 -> 32 72 / 65, 32 -> 64 -> 32 73 / 66; 64 -> 64 -> 64 2^18
  // 35.2 / 33.9), but not in the largest ones where both are wide or the output is off 16 bytes (2^20 rows 48 -> 64 -> 32 90 / 93, 32 -> 64 -> 64 76 / 78,
  // 64 -> 64 -> 64 102 / 112, 2^19 53 / 56; 32 -> 64 -> 20 76 / 79, 2^19 44.0 / 44.6).
  const bool many = depth == 2 ? g.n > 1 << 16 : out <= 16 && g.n > 1 << 19;
  if (many && wt != at::kFloat && depth <= 2 && H == 64 && in <= 64 && out <= 64 && (decoder || m.x.scalar_type() == wt) && in % 4 == 0 && out % 4 == 0 &&
      relu) {
    // The weight gradients come back summed in a fixed order, in one uninitialised buffer (no clearing, no cast
    // kernel).  The buffer is the call's own: its pieces become the .grad tensors.
    const Pieces at(m.w, 8);
    flat = at::empty({at.total}, float_grads ? m.w[0].options().dtype(at::kFloat) : m.w[0].options());
    const int64_t bytes = nf_mlp_bwd_rounded_workspace_bytes(in, H, out);
    const Tensor ws = scratch(bytes, m.x);
    if (need_dx) dx = at::empty(m.x.sizes(), m.x.options());
    const int rc = nf_mlp_bwd_summed(x.p, x.stride, g.p, g.stride, ptr(dx), in, ptr(m.w[0]), ptr(m.w[1]), ptr(m.w[4]), ptr(m.w[5]), ptr(m.w[2]),
                                      ptr(m.w[3]), at.at(flat, m.w[0], 0), at.at(flat, m.w[1], 1), at.at(flat, m.w[4], 4), at.at(flat, m.w[5], 5),
                                     at.at(flat, m.w[2], 2), at.at(flat, m.w[3], 3), x.n, in, H, out, depth, m.act, dt,
                                     code_of(m.x.scalar_type()), float_grads ? NF_F32 : dt, ptr(ws), bytes, stream_of(m.x));
    if (rc != NF_EUNSUPPORTED) {  // unsupported: rows off 8-byte boundaries, the general path below takes them
      check(rc, "nf_mlp_bwd_summed");
      return finish(at, flat);
    }
  }
  if (whole_bytes > 0) {
    const Pieces at(m.w, 8);
    flat = at::empty({at.total}, float_grads ? m.w[0].options().dtype(at::kFloat) : m.w[0].options());
    const Tensor ws = scratch(whole_bytes, m.x);
    dx = need_dx ? at::empty(m.x.sizes(), m.x.options()) : Tensor();
    check(nf_mlp_bwd_whole(x.p, x.stride, g.p, g.stride, ptr(dx), in, ptr(m.w[0]), ptr(m.w[1]), ptr(m.w[4]), ptr(m.w[5]), ptr(m.w[2]), ptr(m.w[3]),
                           at.at(flat, m.w[0], 0), at.at(flat, m.w[1], 1), at.at(flat, m.w[4], 4), at.at(flat, m.w[5], 5), at.at(flat, m.w[2], 2),
                           at.at(flat, m.w[3], 3), x.n, in, H, out, depth, m.act, dt, code_of(m.x.scalar_type()), float_grads ? NF_F32 : dt, ptr(ws),
                           whole_bytes, stream_of(m.x)),
          "nf_mlp_bwd_whole");
    return finish(at, flat);
  }
  const Pieces at(m.w, 4);
  const int64_t bytes = nf_mlp_workspace_bytes(g.n, H, depth, m.act, 1, dt);
  // float32 networks of one and two hidden layers: the gradients are written, with no fill in front (32 -> 64 -> 64 -> 16, 100003 rows: forward and backward 84 -> 78 us)
  const bool written = wt == at::kFloat && depth <= 2 && g.n > 0;
  flat = written ? at::empty({at.total}, m.w[0].options()) : at::zeros({at.total}, m.w[0].options().dtype(at::kFloat));
  const Tensor ws = scratch(bytes, m.x);
  dx = need_dx ? at::empty(m.x.sizes(), m.x.options()) : Tensor();
  const auto grad = [&](int i) { return (float*)at.at(flat, m.w[i], i); };
  if (written) {
    const auto f = [](const void* p) { return (const float*)p; };
    check(nf_mlp_bwd_f32(f(x.p), x.stride, f(g.p), g.stride, (float*)ptr(dx), in, f(ptr(m.w[0])), f(ptr(m.w[1])), f(ptr(m.w[4])), f(ptr(m.w[5])),
                         f(ptr(m.w[2])), f(ptr(m.w[3])), grad(0), grad(1), grad(4), grad(5), grad(2), grad(3), x.n, in, H, out, depth, m.act, ptr(ws),
                         bytes, stream_of(m.x)),
          "nf_mlp_bwd_f32");
    return finish(at, flat);
  }
  check(nf_mlp_bwd(x.p, x.stride, g.p, g.stride, ptr(dx), in, ptr(m.w[0]), ptr(m.w[1]), ptr(m.w[4]), ptr(m.w[5]), ptr(m.w[2]), ptr(m.w[3]), grad(0),
                   grad(1), grad(4), grad(5), grad(2), grad(3), x.n, in, H, out, depth, m.act, dt, code_of(m.x.scalar_type()), ptr(ws), bytes,
                   stream_of(m.x)),
        "nf_mlp_bwd");
  // float32 accumulators, rounded once to the parameters' dtype (one kernel for all of them)
  return finish(at, float_grads || wt == at::kFloat ? flat : flat.to(wt));
}

// x and the parameters in float16 (autocast)
void cast_half(Mlp& m) {
  m.x = m.x.to(at::kHalf);
  bool floats = true;
  for (const Tensor& t : m.w) floats = floats && (!t.defined() || (t.scalar_type() == at::kFloat && t.is_contiguous()));
  if (!floats) {
    for (Tensor& t : m.w)
      if (t.defined()) t = t.to(at::kHalf);
    return;
  }
  const c10::DeviceGuard guard(m.x.device());
  const Pieces at(m.w, 8);
  const Tensor flat = at::empty({at.total}, m.w[0].options().dtype(at::kHalf));
  const float* src[6];
  int64_t count[6];
  int n = 0;
  for (const Tensor& t : m.w)
    if (t.defined()) {
      src[n] = (const float*)t.data_ptr();
      count[n++] = t.numel();
    }
  check(nf_cast_pieces_f16(src, count, n, flat.data_ptr(), stream_of(flat)), "nf_cast_pieces_f16");
  for (int i = 0; i < 6; ++i) m.w[i] = at.view(flat, m.w[i], i);
}

struct FusedMlp : torch::autograd::Function<FusedMlp> {
  // half: autocast to float16 -- what is not float16 is cast, and the parameters' gradients go back as float32
  static Tensor forward(AutogradContext* ctx, Tensor x, Tensor w_in, std::optional<Tensor> b_in, Tensor w_out, std::optional<Tensor> b_out,
                        std::optional<Tensor> w_hid, std::optional<Tensor> b_hid, int64_t act, bool half) {
    Mlp m{x, {w_in, b_in.value_or(Tensor()), w_out, b_out.value_or(Tensor()), w_hid.value_or(Tensor()), b_hid.value_or(Tensor())}, (int)act};
    const bool float_grads = half && w_in.scalar_type() == at::kFloat;
    const at::AutoDispatchBelowADInplaceOrView below;
    if (half) cast_half(m);
    ctx->save_for_backward({m.x, m.w[0], m.w[1], m.w[2], m.w[3], m.w[4], m.w[5]});
    ctx->saved_data["act"] = act;
    ctx->saved_data["float_grads"] = float_grads;
    return mlp_forward(std::move(m));
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::AutoDispatchBelowADInplaceOrView below;
    variable_list r = mlp_backward(Mlp{s[0], {s[1], s[2], s[3], s[4], s[5], s[6]}, (int)ctx->saved_data["act"].toInt()}, grads[0],
                                   ctx->needs_input_grad(0), ctx->saved_data["float_grads"].toBool());
    r.resize(9);
    return r;
  }
};

// ------------------------------------------------------------------------------------------------ reversible MLP
Tensor reversible_forward(const Tensor& x, std::array<Tensor, 4> w, int act) {
  const c10::DeviceGuard guard(x.device());
  for (Tensor& t : w) t = contiguous(t);
  const int64_t width = x.size(-1), H = width / 2;
  const Rows r(x, width);
  Tensor y = at::empty(x.sizes(), x.options());
  check(nf_revmlp_fwd(r.p, r.stride, y.data_ptr(), width, ptr(w[0]), ptr(w[1]), ptr(w[2]), ptr(w[3]), r.n, (int)H, (int)(w[0].size(0) / (2 * H)), act,
                      code_of(x.scalar_type()), stream_of(x)),
        "nf_revmlp_fwd");
  return y;
}

// (dx, dw1, db1, dw2, db2)
variable_list reversible_backward(const Tensor& y, Tensor dy, std::array<Tensor, 4> w, int act, bool float_grads) {
  const c10::DeviceGuard guard(y.device());
  for (Tensor& t : w) t = contiguous(t);
  if (dy.scalar_type() != y.scalar_type()) dy = dy.to(y.scalar_type());
  const int64_t width = y.size(-1), H = width / 2;
  const Rows ry(y, width), rd(dy, width);
  const Tensor dx = at::empty(y.sizes(), y.options()), x_rec = at::empty(y.sizes(), y.options());
  const Pieces at(w, 8);
  const int dt = code_of(y.scalar_type()), blocks = (int)(w[0].size(0) / (2 * H));
  const auto options = float_grads ? y.options().dtype(at::kFloat) : y.options();
  const Tensor f = ry.n > 0 ? at::empty({at.total}, options) : at::zeros({at.total}, options);
  if (ry.n > 0) {
    const int64_t bytes = nf_revmlp_bwd_workspace_bytes(ry.n, (int)H, blocks);
    const Tensor ws = scratch(bytes, y);
    check(nf_revmlp_bwd_summed(ry.p, ry.stride, rd.p, rd.stride, dx.data_ptr(), width, x_rec.data_ptr(), width, ptr(w[0]), ptr(w[1]), ptr(w[2]), ptr(w[3]),
                               at.at(f, w[0], 0), at.at(f, w[1], 1), at.at(f, w[2], 2), at.at(f, w[3], 3), ry.n, (int)H, blocks, act, dt,
                               float_grads ? NF_F32 : dt, ptr(ws), bytes, stream_of(y)),
          "nf_revmlp_bwd_summed");
  }
  return {dx, at.view(f, w[0], 0), at.view(f, w[1], 1), at.view(f, w[2], 2), at.view(f, w[3], 3)};
}

struct ReversibleMlp : torch::autograd::Function<ReversibleMlp> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, Tensor w1, std::optional<Tensor> b1, Tensor w2, std::optional<Tensor> b2, int64_t act) {
    const at::AutoDispatchBelowADInplaceOrView below;
    const std::array<Tensor, 4> w{w1, b1.value_or(Tensor()), w2, b2.value_or(Tensor())};
    const Tensor y = reversible_forward(x, w, (int)act);
    ctx->save_for_backward({y, w[0], w[1], w[2], w[3]});  // the output, not the input
    ctx->saved_data["act"] = act;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::AutoDispatchBelowADInplaceOrView below;
    variable_list r = reversible_backward(s[0], grads[0], {s[1], s[2], s[3], s[4]}, (int)ctx->saved_data["act"].toInt(), false);
    r.resize(6);
    return r;
  }
};

// ------------------------------------------------------------------------------------------------ Python
// A plain GPU tensor: no subclass, no wrapper of a function transform, no tangent of a forward-mode derivative (the kernels have no
// such derivative: the autograd Function refuses it), a floating type the kernels know.
bool plain(PyObject* o, Tensor* t) {
  if (!THPVariable_CheckTypeExact(Py_TYPE(o))) return false;
  *t = THPVariable_Unpack(o);
  const auto keys = t->key_set();
  return t->is_cuda() && t->layout() == at::kStrided && !keys.has(c10::DispatchKey::FuncTorchBatched) &&
         !keys.has(c10::DispatchKey::FuncTorchGradWrapper) && !keys.has(c10::DispatchKey::Functionalize) && !keys.has(c10::DispatchKey::Python) &&
         !t->is_conj() && !t->is_neg() && !t->_fw_grad(/*level=*/0).defined();
}

bool plain_or_none(PyObject* o, std::optional<Tensor>* t) {
  if (o == Py_None) return true;
  Tensor v;
  if (!plain(o, &v)) return false;
  *t = std::move(v);
  return true;
}

// A dispatch or function mode, a function transform (vmap, grad, jvp: the autograd Functions refuse them), or the tracer, which records
// an autograd Function but would see nothing of a launch made here.
bool modes_active() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() || torch::jit::tracer::isTracing() ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

bool autocast() { return at::autocast::is_autocast_enabled(at::kCUDA); }

bool as_int(PyObject* o, int64_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

bool as_double(PyObject* o, double* v) {
  if (!PyFloat_CheckExact(o) && !PyLong_CheckExact(o)) return false;
  *v = PyFloat_AsDouble(o);
  if (*v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

int activation(PyObject* o, bool gelu) {
  if (!PyUnicode_Check(o)) return -1;
  const char* s = PyUnicode_AsUTF8(o);
  if (s == nullptr) {
    PyErr_Clear();
    return -1;
  }
  if (!strcmp(s, "relu")) return NF_ACT_RELU;
  if (!strcmp(s, "silu")) return NF_ACT_SILU;
  if (!strcmp(s, "relu2")) return NF_ACT_RELU2;
  if (!strcmp(s, "none")) return NF_ACT_NONE;
  return gelu && !strcmp(s, "gelu") ? NF_ACT_GELU : -1;
}

PyObject* wrap(const Tensor& t) { return THPVariable_Wrap(t); }

PyObject* wrap_list(const variable_list& v) {
  PyObject* r = PyTuple_New((Py_ssize_t)v.size());
  if (r == nullptr) return nullptr;
  for (size_t i = 0; i < v.size(); ++i) {
    PyObject* o = v[i].defined() ? wrap(v[i]) : Py_NewRef(Py_None);
    if (o == nullptr) {
      Py_DECREF(r);
      return nullptr;
    }
    PyTuple_SET_ITEM(r, (Py_ssize_t)i, o);
  }
  return r;
}

Tensor tensor_arg(PyObject* o) { return o == Py_None ? Tensor() : THPVariable_Unpack(o); }

#define NARGS(k) TORCH_CHECK(n == (k), "expected ", (k), " arguments, got ", n)

// add_geometry(T, levels, D, F, min_res, max_res, address of a nf_hash_geom, rows)
PyObject* add_geometry(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NARGS(8);
  std::array<int64_t, 8> v{};
  for (int i = 0; i < 8; ++i) TORCH_CHECK(as_int(a[i], &v[i]), "integer arguments expected");
  auto e = std::make_unique<Geometry>();
  for (int i = 0; i < 6; ++i) e->key[i] = v[i];
  e->g = *(const nf_hash_geom*)(uintptr_t)v[6];
  e->rows = v[7];
  if (find_geometry(e->key) == nullptr && geometries().size() < MAX_GEOMETRIES) geometries().push_back(std::move(e));
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// hash_encoding(coord, embeddings, features, pi, T, min_res, max_res, levels, divider, bwd_divider, scale, flags)
PyObject* hash_encoding(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NARGS(12);
  Tensor coords, table;
  std::optional<Tensor> pi;
  int64_t T, lo, hi, levels, flags;
  double scale;
  if (modes_active() || autocast() || !plain(a[0], &coords) || !plain(a[1], &table) || a[2] != Py_None || !plain_or_none(a[3], &pi) ||
      !as_int(a[4], &T) || !as_int(a[5], &lo) || !as_int(a[6], &hi) || !as_int(a[7], &levels) || a[8] != Py_None || a[9] != Py_None ||
      !as_double(a[10], &scale) || !as_int(a[11], &flags))
    Py_RETURN_NONE;
  if (coords.dim() < 1 || table.dim() != 2 || code_of(coords.scalar_type()) < 0 || code_of(table.scalar_type()) < 0 || coords.requires_grad() ||
      coords.device() != table.device() || !table.is_contiguous())
    Py_RETURN_NONE;
  const int64_t D = coords.size(-1);
  const Geometry* geo = find_geometry({T, levels, D, table.size(1), lo, hi});
  if (geo == nullptr || table.size(0) < geo->rows || (D > 3 && !pi)) Py_RETURN_NONE;
  if (pi && (pi->scalar_type() != at::kLong || pi->dim() != 1 || pi->numel() < D || !pi->is_contiguous() || pi->device() != coords.device()))
    Py_RETURN_NONE;
  Tensor out;
  {
    pybind11::gil_scoped_release release;
    const Tensor primes = pi ? *pi : default_primes(coords.device());
    if (at::GradMode::is_enabled() && table.requires_grad()) {
      out = HashEncoding::apply(coords, table, primes, geo, scale, flags);
    } else {
      const at::AutoDispatchBelowADInplaceOrView below;
      out = encode_forward(coords, table, primes, *geo, scale, flags);
    }
  }
  return wrap(out);
  END_HANDLE_TH_ERRORS
}

// primes(index of a GPU): the default primes there
PyObject* primes(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NARGS(1);
  int64_t index;
  TORCH_CHECK(as_int(a[0], &index) && index >= 0 && index < c10::hip::device_count(), "index of a GPU expected");
  Tensor t;
  {
    pybind11::gil_scoped_release release;
    t = default_primes(c10::Device(c10::kCUDA, (c10::DeviceIndex)index));
  }
  return wrap(t);
  END_HANDLE_TH_ERRORS
}

// hash_table_grad(coords, grad, de, pi, address of a nf_hash_geom, scale, flags): adds into de
PyObject* hash_table_grad(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NARGS(7);
  const Tensor coords = tensor_arg(a[0]), grad = tensor_arg(a[1]), de = tensor_arg(a[2]), pi = tensor_arg(a[3]);
  int64_t geom, flags;
  double scale;
  TORCH_CHECK(as_int(a[4], &geom) && as_double(a[5], &scale) && as_int(a[6], &flags), "address, scale and flags expected");
  TORCH_CHECK_TYPE(code_of(coords.scalar_type()) >= 0 && code_of(grad.scalar_type()) >= 0, "unsupported dtype; expected float32, float16 or bfloat16");
  {
    pybind11::gil_scoped_release release;
    const at::AutoDispatchBelowADInplaceOrView below;
    encode_backward(coords, grad, de, pi, *(const nf_hash_geom*)(uintptr_t)geom, scale, flags);
  }
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

bool mlp_fits(const Tensor& x, const std::array<Tensor, 6>& w, bool cast) {
  if (x.dim() != 3 || w[0].dim() != 2 || w[2].dim() != 2) return false;
  const int64_t H = w[0].size(0), in = w[0].size(1), out = w[2].size(0);
  if (in != x.size(2) || w[2].size(1) != H || in > 64 || H > 64 || out > 64 || H < 16 || (H & (H - 1)) != 0 || in < 1 || out < 1) return false;
  if (w[1].defined() && (w[1].dim() != 1 || w[1].size(0) != H)) return false;
  if (w[3].defined() && (w[3].dim() != 1 || w[3].size(0) != out)) return false;
  if (w[4].defined()) {
    if (w[4].dim() != 2 || w[4].size(0) < H || w[4].size(0) % H != 0 || w[4].size(1) != H) return false;
    if (w[5].defined() && (w[5].dim() != 2 || w[5].size(0) != w[4].size(0) / H || w[5].size(1) != H)) return false;
  } else if (w[5].defined()) {
    return false;
  }
  const int xt = code_of(x.scalar_type()), wt = code_of(w[0].scalar_type());
  if (xt < 0 || wt < 0 || (!cast && (xt == NF_F32) != (wt == NF_F32))) return false;
  for (const Tensor& t : w)
    if (t.defined() && (t.scalar_type() != w[0].scalar_type() || t.device() != x.device())) return false;
  return true;
}

// mlp(x, w_in, b_in, w_out, b_out, w_hid, b_hid, activation)
PyObject* mlp(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NARGS(8);
  Tensor x, w_in, w_out;
  std::optional<Tensor> b_in, b_out, w_hid, b_hid;
  const int act = activation(a[7], false);
  if (modes_active() || act < 0 || !plain(a[0], &x) || !plain(a[1], &w_in) || !plain_or_none(a[2], &b_in) || !plain(a[3], &w_out) ||
      !plain_or_none(a[4], &b_out) || !plain_or_none(a[5], &w_hid) || !plain_or_none(a[6], &b_hid))
    Py_RETURN_NONE;
  const bool cast = autocast();
  const std::array<Tensor, 6> w{w_in, b_in.value_or(Tensor()), w_out, b_out.value_or(Tensor()), w_hid.value_or(Tensor()), b_hid.value_or(Tensor())};
  if (!mlp_fits(x, w, cast)) Py_RETURN_NONE;
  bool grad = x.requires_grad();
  for (const Tensor& t : w) grad = grad || (t.defined() && t.requires_grad());
  Tensor y;
  {
    pybind11::gil_scoped_release release;
    if (at::GradMode::is_enabled() && grad) {
      y = FusedMlp::apply(x, w_in, b_in, w_out, b_out, w_hid, b_hid, (int64_t)act, cast);
    } else {
      const at::AutoDispatchBelowADInplaceOrView below;
      Mlp m{x, w, act};
      if (cast) cast_half(m);
      y = mlp_forward(std::move(m));
    }
  }
  return wrap(y);
  END_HANDLE_TH_ERRORS
}

Mlp mlp_args(PyObject* const* a, PyObject* act) {
  int64_t code;
  TORCH_CHECK(as_int(act, &code), "activation code expected");
  Mlp m{tensor_arg(a[0]), {}, (int)code};
  for (int i = 0; i < 6; ++i) m.w[i] = tensor_arg(a[1 + i]);
  return m;
}

// mlp_launch_forward(x, w_in, b_in, w_out, b_out, w_hid, b_hid, activation code) on checked arguments
PyObject* mlp_launch_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NARGS(8);
  Mlp m = mlp_args(a, a[7]);
  Tensor y;
  {
    pybind11::gil_scoped_release release;
    const at::AutoDispatchBelowADInplaceOrView below;
    y = mlp_forward(std::move(m));
  }
  return wrap(y);
  END_HANDLE_TH_ERRORS
}

// mlp_launch_backward(x, w_in, b_in, w_out, b_out, w_hid, b_hid, activation code, dy, need_dx, float_grads)
PyObject* mlp_launch_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NARGS(11);
  Mlp m = mlp_args(a, a[7]);
  const Tensor dy = tensor_arg(a[8]);
  const bool need_dx = a[9] == Py_True, float_grads = a[10] == Py_True;
  variable_list r;
  {
    pybind11::gil_scoped_release release;
    const at::AutoDispatchBelowADInplaceOrView below;
    r = mlp_backward(std::move(m), dy, need_dx, float_grads);
  }
  return wrap_list(r);
  END_HANDLE_TH_ERRORS
}

// reversible(x, w1, b1, w2, b2, activation)
PyObject* reversible(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NARGS(6);
  Tensor x, w1, w2;
  std::optional<Tensor> b1, b2;
  const int act = activation(a[5], true);
  if (modes_active() || autocast() || act < 0 || !plain(a[0], &x) || !plain(a[1], &w1) || !plain_or_none(a[2], &b1) || !plain(a[3], &w2) ||
      !plain_or_none(a[4], &b2))
    Py_RETURN_NONE;
  const auto dt = x.scalar_type();
  if ((dt != at::kHalf && dt != at::kBFloat16) || x.dim() < 1 || x.size(-1) < 2 || x.size(-1) % 2 != 0 || x.size(-1) > 128) Py_RETURN_NONE;
  const int64_t H = x.size(-1) / 2;
  if (w1.dim() != 2 || w1.size(1) != H || w1.size(0) < 2 * H || w1.size(0) % (2 * H) != 0 || w2.sizes() != w1.sizes()) Py_RETURN_NONE;
  const std::array<Tensor, 4> w{w1, b1.value_or(Tensor()), w2, b2.value_or(Tensor())};
  bool grad = x.requires_grad();
  for (int i = 0; i < 4; ++i) {
    if (!w[i].defined()) continue;
    if (w[i].scalar_type() != dt || w[i].device() != x.device()) Py_RETURN_NONE;
    if (i % 2 == 1 && (w[i].dim() != 2 || w[i].size(0) != w1.size(0) / H || w[i].size(1) != H)) Py_RETURN_NONE;
    grad = grad || w[i].requires_grad();
  }
  Tensor y;
  {
    pybind11::gil_scoped_release release;
    if (at::GradMode::is_enabled() && grad) {
      y = ReversibleMlp::apply(x, w1, b1, w2, b2, (int64_t)act);
    } else {
      const at::AutoDispatchBelowADInplaceOrView below;
      y = reversible_forward(x, w, act);
    }
  }
  return wrap(y);
  END_HANDLE_TH_ERRORS
}

// reversible_launch_forward(x, w1, b1, w2, b2, activation code) on checked arguments
PyObject* reversible_launch_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NARGS(6);
  int64_t act;
  TORCH_CHECK(as_int(a[5], &act), "activation code expected");
  const Tensor x = tensor_arg(a[0]);
  const std::array<Tensor, 4> w{tensor_arg(a[1]), tensor_arg(a[2]), tensor_arg(a[3]), tensor_arg(a[4])};
  Tensor y;
  {
    pybind11::gil_scoped_release release;
    const at::AutoDispatchBelowADInplaceOrView below;
    y = reversible_forward(x, w, (int)act);
  }
  return wrap(y);
  END_HANDLE_TH_ERRORS
}

// reversible_launch_backward(y, w1, b1, w2, b2, activation code, dy, float_grads)
PyObject* reversible_launch_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  NARGS(8);
  int64_t act;
  TORCH_CHECK(as_int(a[5], &act), "activation code expected");
  const Tensor y = tensor_arg(a[0]), dy = tensor_arg(a[6]);
  const std::array<Tensor, 4> w{tensor_arg(a[1]), tensor_arg(a[2]), tensor_arg(a[3]), tensor_arg(a[4])};
  const bool float_grads = a[7] == Py_True;
  variable_list r;
  {
    pybind11::gil_scoped_release release;
    const at::AutoDispatchBelowADInplaceOrView below;
    r = reversible_backward(y, dy, w, (int)act, float_grads);
  }
  return wrap_list(r);
  END_HANDLE_TH_ERRORS
}

#define ENTRY(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {ENTRY(add_geometry),       ENTRY(primes),                    ENTRY(hash_encoding), ENTRY(hash_table_grad),
                         ENTRY(mlp),                ENTRY(mlp_launch_forward),        ENTRY(mlp_launch_backward),
                         ENTRY(reversible),         ENTRY(reversible_launch_forward), ENTRY(reversible_launch_backward),
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "Host side of the operators (see csrc/host_native.cpp)", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
