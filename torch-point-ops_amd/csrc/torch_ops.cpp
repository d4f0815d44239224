// torch_ops.cpp -- PyTorch operator registrations for torch_point_ops on ROCm.
//
// Registers the reference's operator schemas verbatim
//   torch_point_ops_chamfer  chamfer.cpp:34-39
//   torch_point_ops_knn      knn.cpp:166-171
//   torch_point_ops_fps      fps.cpp:158-162
//   torch_point_ops_quick_fps fps.cpp:165-167
//   torch_point_ops_emd      emd.cpp:31-34
// and implements them for the CUDA dispatch key (HIP tensors on ROCm) by
// calling the C ABI of libtpo_hip.so on the current HIP stream.  Validation
// and error texts follow the reference's TORCH_CHECKs.  The shim does the
// allocation (torch caching allocator); the kernels write every output
// element, so outputs are created with empty().
#include <Python.h>
#include <torch/all.h>
#include <torch/library.h>

#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/autograd/custom_function.h>

#include <tuple>

#include "tpo.h"

namespace torch_point_ops {
namespace {

int dtype_code(const at::Tensor& t, const char* op) {
  switch (t.scalar_type()) {
    case at::kFloat: return TPO_F32;
    case at::kDouble: return TPO_F64;
    case at::kHalf: return TPO_F16;
    default:
      TORCH_CHECK(false, op, " not implemented for '", t.scalar_type(), "'");
  }
  return -1;
}

// A tensor whose data starts on a 16-byte boundary (a copy if it does not).
at::Tensor aligned16(const at::Tensor& t) {
  return ((uintptr_t)t.data_ptr() & 15) ? t.clone(at::MemoryFormat::Contiguous) : t;
}

void* stream_of(const at::Tensor& t) {
  return (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

void check_rc(int rc, const char* op) {
  TORCH_CHECK(rc == TPO_OK, op, " failed: ", tpo_last_error());
}

void check_hip(const at::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be a GPU tensor");
}

// ------------------------------------------------------------------ chamfer
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> chamfer_forward_hip(
    const at::Tensor& xyz1_in, const at::Tensor& xyz2_in) {
  check_hip(xyz1_in, "xyz1");
  check_hip(xyz2_in, "xyz2");
  TORCH_CHECK(xyz1_in.dim() == 3 && xyz2_in.dim() == 3 && xyz1_in.size(2) == 3 &&
                  xyz2_in.size(2) == 3,
              "chamfer_forward expects (B,N,3) and (B,M,3) tensors");
  TORCH_CHECK(xyz1_in.size(0) == xyz2_in.size(0), "batch sizes differ");
  TORCH_CHECK(xyz1_in.scalar_type() == xyz2_in.scalar_type(), "dtypes differ");
  TORCH_CHECK(xyz1_in.device() == xyz2_in.device(), "xyz1 and xyz2 must be on the same device");
  c10::OptionalDeviceGuard guard(xyz1_in.device());
  const at::Tensor xyz1 = xyz1_in.contiguous(), xyz2 = xyz2_in.contiguous();
  const int64_t B = xyz1.size(0), N = xyz1.size(1), M = xyz2.size(1);
  const int dt = dtype_code(xyz1, "chamfer_forward");
  at::Tensor dist1 = at::empty({B, N}, xyz1.options());
  at::Tensor dist2 = at::empty({B, M}, xyz1.options());
  at::Tensor idx1 = at::empty({B, N}, xyz1.options().dtype(at::kInt));
  at::Tensor idx2 = at::empty({B, M}, xyz1.options().dtype(at::kInt));
  const int64_t ws_bytes = tpo_chamfer_workspace_size(dt, B, N, M);
  at::Tensor ws;
  if (ws_bytes > 0) ws = at::empty({ws_bytes}, xyz1.options().dtype(at::kByte));
  check_rc(tpo_chamfer_fwd(dt, xyz1.data_ptr(), xyz2.data_ptr(), B, N, M, dist1.data_ptr(),
                           dist2.data_ptr(), idx1.data_ptr<int32_t>(), idx2.data_ptr<int32_t>(),
                           ws_bytes > 0 ? ws.data_ptr() : nullptr, ws_bytes, stream_of(xyz1)),
           "chamfer_forward");
  return {dist1, dist2, idx1, idx2};
}

std::tuple<at::Tensor, at::Tensor> chamfer_backward_hip(
    const at::Tensor& xyz1_in, const at::Tensor& xyz2_in, const at::Tensor& idx1_in,
    const at::Tensor& idx2_in, const at::Tensor& gd1_in, const at::Tensor& gd2_in) {
  check_hip(xyz1_in, "xyz1");
  c10::OptionalDeviceGuard guard(xyz1_in.device());
  const at::Tensor xyz1 = xyz1_in.contiguous(), xyz2 = xyz2_in.contiguous();
  const int64_t B = xyz1.size(0), N = xyz1.size(1), M = xyz2.size(1);
  TORCH_CHECK(idx1_in.scalar_type() == at::kInt && idx2_in.scalar_type() == at::kInt,
              "chamfer_backward expects int32 indices");
  TORCH_CHECK(idx1_in.numel() == B * N && idx2_in.numel() == B * M, "index shapes differ");
  TORCH_CHECK(gd1_in.numel() == B * N && gd2_in.numel() == B * M, "grad shapes differ");
  const at::Tensor idx1 = idx1_in.contiguous(), idx2 = idx2_in.contiguous();
  const at::Tensor gd1 = gd1_in.to(xyz1.scalar_type()).contiguous();
  const at::Tensor gd2 = gd2_in.to(xyz1.scalar_type()).contiguous();
  const int dt = dtype_code(xyz1, "chamfer_backward");
  at::Tensor g1 = at::empty_like(xyz1), g2 = at::empty_like(xyz2);
  check_rc(tpo_chamfer_bwd(dt, xyz1.data_ptr(), xyz2.data_ptr(), idx1.data_ptr<int32_t>(),
                           idx2.data_ptr<int32_t>(), gd1.data_ptr(), gd2.data_ptr(), B, N, M,
                           g1.data_ptr(), g2.data_ptr(), stream_of(xyz1)),
           "chamfer_backward");
  return {g1, g2};
}

// ChamferDistance(reduction="mean" / "sum") fused: loss and the indices the
// backward needs (chamfer.py:18-24 reduces chamfer_forward's distances).
std::tuple<at::Tensor, at::Tensor, at::Tensor> chamfer_loss_forward_hip(
    const at::Tensor& xyz1_in, const at::Tensor& xyz2_in, bool mean) {
  check_hip(xyz1_in, "xyz1");
  check_hip(xyz2_in, "xyz2");
  TORCH_CHECK(xyz1_in.dim() == 3 && xyz2_in.dim() == 3 && xyz1_in.size(2) == 3 &&
                  xyz2_in.size(2) == 3,
              "chamfer_loss_forward expects (B,N,3) and (B,M,3) tensors");
  TORCH_CHECK(xyz1_in.size(0) == xyz2_in.size(0), "batch sizes differ");
  TORCH_CHECK(xyz1_in.scalar_type() == xyz2_in.scalar_type(), "dtypes differ");
  TORCH_CHECK(xyz1_in.device() == xyz2_in.device(), "xyz1 and xyz2 must be on the same device");
  c10::OptionalDeviceGuard guard(xyz1_in.device());
  const at::Tensor xyz1 = xyz1_in.contiguous(), xyz2 = xyz2_in.contiguous();
  const int64_t B = xyz1.size(0), N = xyz1.size(1), M = xyz2.size(1);
  const int dt = dtype_code(xyz1, "chamfer_loss_forward");
  at::Tensor loss = at::empty({}, xyz1.options());
  at::Tensor idx1 = at::empty({B, N}, xyz1.options().dtype(at::kInt));
  at::Tensor idx2 = at::empty({B, M}, xyz1.options().dtype(at::kInt));
  const int64_t ws_bytes = tpo_chamfer_loss_workspace_size(dt, B, N, M);
  TORCH_CHECK(ws_bytes >= 0, "chamfer_loss_forward: bad sizes");
  at::Tensor ws = at::empty({std::max<int64_t>(ws_bytes, 1)}, xyz1.options().dtype(at::kByte));
  check_rc(tpo_chamfer_loss_fwd(dt, xyz1.data_ptr(), xyz2.data_ptr(), B, N, M, mean ? 1 : 0,
                                loss.data_ptr(), idx1.data_ptr<int32_t>(),
                                idx2.data_ptr<int32_t>(), ws.data_ptr(), ws_bytes,
                                stream_of(xyz1)),
           "chamfer_loss_forward");
  return {loss, idx1, idx2};
}

std::tuple<at::Tensor, at::Tensor> chamfer_loss_backward_hip(
    const at::Tensor& xyz1_in, const at::Tensor& xyz2_in, const at::Tensor& idx1_in,
    const at::Tensor& idx2_in, const at::Tensor& grad_loss_in, bool mean) {
  check_hip(xyz1_in, "xyz1");
  c10::OptionalDeviceGuard guard(xyz1_in.device());
  const at::Tensor xyz1 = xyz1_in.contiguous(), xyz2 = xyz2_in.contiguous();
  const int64_t B = xyz1.size(0), N = xyz1.size(1), M = xyz2.size(1);
  TORCH_CHECK(idx1_in.scalar_type() == at::kInt && idx2_in.scalar_type() == at::kInt,
              "chamfer_loss_backward expects int32 indices");
  TORCH_CHECK(idx1_in.numel() == B * N && idx2_in.numel() == B * M, "index shapes differ");
  TORCH_CHECK(grad_loss_in.numel() == 1, "chamfer_loss_backward expects a scalar gradient");
  const at::Tensor idx1 = idx1_in.contiguous(), idx2 = idx2_in.contiguous();
  const at::Tensor gl = grad_loss_in.to(xyz1.device(), xyz1.scalar_type()).contiguous();
  const int dt = dtype_code(xyz1, "chamfer_loss_backward");
  at::Tensor g1 = at::empty_like(xyz1), g2 = at::empty_like(xyz2);
  check_rc(tpo_chamfer_loss_bwd(dt, xyz1.data_ptr(), xyz2.data_ptr(), idx1.data_ptr<int32_t>(),
                                idx2.data_ptr<int32_t>(), gl.data_ptr(), mean ? 1 : 0, B, N, M,
                                g1.data_ptr(), g2.data_ptr(), stream_of(xyz1)),
           "chamfer_loss_backward");
  return {g1, g2};
}

// Autograd of the fused module loss, in C++: the step's backward runs no
// Python (the module's gradient is the hot path of ChamferDistance training).
// Index outputs are non-differentiable and their gradients not materialised.
class ChamferLossFunction : public torch::autograd::Function<ChamferLossFunction> {
 public:
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx,
                                                const at::Tensor& xyz1, const at::Tensor& xyz2,
                                                bool mean) {
    static auto op = c10::Dispatcher::singleton()
                         .findSchemaOrThrow("torch_point_ops_chamfer::chamfer_loss_forward", "")
                         .typed<std::tuple<at::Tensor, at::Tensor, at::Tensor>(
                             const at::Tensor&, const at::Tensor&, bool)>();
    at::Tensor loss, idx1, idx2;
    {
      at::AutoDispatchBelowADInplaceOrView below;
      std::tie(loss, idx1, idx2) = op.call(xyz1, xyz2, mean);
    }
    ctx->save_for_backward({xyz1, xyz2, idx1, idx2});
    ctx->saved_data["mean"] = mean;
    ctx->mark_non_differentiable({idx1, idx2});
    ctx->set_materialize_grads(false);
    return {loss, idx1, idx2};
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    static auto op = c10::Dispatcher::singleton()
                         .findSchemaOrThrow("torch_point_ops_chamfer::chamfer_loss_backward", "")
                         .typed<std::tuple<at::Tensor, at::Tensor>(
                             const at::Tensor&, const at::Tensor&, const at::Tensor&,
                             const at::Tensor&, const at::Tensor&, bool)>();
    if (!grads[0].defined()) return {at::Tensor(), at::Tensor(), at::Tensor()};
    const auto saved = ctx->get_saved_variables();
    at::Tensor g1, g2;
    std::tie(g1, g2) = op.call(saved[0], saved[1], saved[2], saved[3], grads[0],
                               ctx->saved_data["mean"].toBool());
    return {g1, g2, at::Tensor()};
  }
};

std::tuple<at::Tensor, at::Tensor, at::Tensor> chamfer_loss_forward_autograd(
    const at::Tensor& xyz1, const at::Tensor& xyz2, bool mean) {
  auto out = ChamferLossFunction::apply(xyz1, xyz2, mean);
  return {out[0], out[1], out[2]};
}

// Whether autograd has to follow the call.  Without it the operator runs as it
// is, also under transforms that a C++ autograd function refuses.
bool followed(const at::Tensor& a) { return at::GradMode::is_enabled() && a.requires_grad(); }

// chamfer_forward's autograd (chamfer/__init__.py:6-28) in C++: an unused
// distance output's gradient arrives undefined and counts as zeros.
class ChamferFunction : public torch::autograd::Function<ChamferFunction> {
 public:
  typedef std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> Outputs;
  static auto op() {
    static auto h = c10::Dispatcher::singleton()
                        .findSchemaOrThrow("torch_point_ops_chamfer::chamfer_forward", "")
                        .typed<Outputs(const at::Tensor&, const at::Tensor&)>();
    return h;
  }
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx,
                                                const at::Tensor& xyz1, const at::Tensor& xyz2) {
    at::Tensor d1, d2, i1, i2;
    {
      at::AutoDispatchBelowADInplaceOrView below;
      std::tie(d1, d2, i1, i2) = op().call(xyz1, xyz2);
    }
    ctx->save_for_backward({xyz1, xyz2, i1, i2});
    ctx->mark_non_differentiable({i1, i2});
    ctx->set_materialize_grads(false);
    return {d1, d2, i1, i2};
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    static auto bwd = c10::Dispatcher::singleton()
                          .findSchemaOrThrow("torch_point_ops_chamfer::chamfer_backward", "")
                          .typed<std::tuple<at::Tensor, at::Tensor>(
                              const at::Tensor&, const at::Tensor&, const at::Tensor&,
                              const at::Tensor&, const at::Tensor&, const at::Tensor&)>();
    if (!grads[0].defined() && !grads[1].defined()) return {at::Tensor(), at::Tensor()};
    const auto s = ctx->get_saved_variables();
    const auto like = [&](const at::Tensor& g, const at::Tensor& idx) {
      return g.defined() ? g : at::zeros_symint(idx.sym_sizes(), s[0].options());
    };
    at::Tensor g1, g2;
    std::tie(g1, g2) = bwd.call(s[0], s[1], s[2], s[3], like(grads[0], s[2]), like(grads[1], s[3]));
    return {g1, g2};
  }
};

ChamferFunction::Outputs chamfer_forward_autograd(const at::Tensor& xyz1, const at::Tensor& xyz2) {
  if (!followed(xyz1) && !followed(xyz2)) {
    at::AutoDispatchBelowADInplaceOrView below;
    return ChamferFunction::op().call(xyz1, xyz2);
  }
  auto out = ChamferFunction::apply(xyz1, xyz2);
  return {out[0], out[1], out[2], out[3]};
}

// chamfer.cpp:21-31: the reference has no CPU kernel.
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> chamfer_forward_cpu(
    const at::Tensor&, const at::Tensor&) {
  TORCH_CHECK(false, "chamfer_forward is not implemented for CPU");
}
std::tuple<at::Tensor, at::Tensor> chamfer_backward_cpu(const at::Tensor&, const at::Tensor&,
                                                        const at::Tensor&, const at::Tensor&,
                                                        const at::Tensor&, const at::Tensor&) {
  TORCH_CHECK(false, "chamfer_backward is not implemented for CPU");
}
std::tuple<at::Tensor, at::Tensor, at::Tensor> chamfer_loss_forward_cpu(const at::Tensor&,
                                                                        const at::Tensor&, bool) {
  TORCH_CHECK(false, "chamfer_forward is not implemented for CPU");
}
std::tuple<at::Tensor, at::Tensor> chamfer_loss_backward_cpu(const at::Tensor&, const at::Tensor&,
                                                             const at::Tensor&, const at::Tensor&,
                                                             const at::Tensor&, bool) {
  TORCH_CHECK(false, "chamfer_backward is not implemented for CPU");
}

// ---------------------------------------------------------------------- knn
std::tuple<at::Tensor, at::Tensor> knn_forward_hip(const at::Tensor& p1_in,
                                                   const at::Tensor& p2_in,
                                                   const at::Tensor& lengths1_in,
                                                   const at::Tensor& lengths2_in, int64_t norm,
                                                   int64_t K, int64_t version) {
  // knn.cu:305-320
  TORCH_CHECK(p1_in.device() == p2_in.device(), "p1 and p2 must be on the same device");
  TORCH_CHECK(p1_in.device() == lengths1_in.device(),
              "p1 and lengths1 must be on the same device");
  TORCH_CHECK(p1_in.device() == lengths2_in.device(),
              "p1 and lengths2 must be on the same device");
  check_hip(p1_in, "p1");
  c10::OptionalDeviceGuard guard(p1_in.device());
  TORCH_CHECK(p1_in.dim() == 3 && p2_in.dim() == 3, "knn_forward expects (N,P,D) tensors");
  const int64_t N = p1_in.size(0), P1 = p1_in.size(1), P2 = p2_in.size(1), D = p1_in.size(2);
  TORCH_CHECK((norm == 1) || (norm == 2), "Norm must be 1 or 2.");
  TORCH_CHECK(p2_in.size(2) == D, "Point sets must have the same last dimension");
  TORCH_CHECK(K >= 0, "K must be non-negative");
  auto idxs = at::empty({N, P1, K}, lengths1_in.options().dtype(at::kLong));
  auto dists = at::empty({N, P1, K}, p1_in.options());
  if (idxs.numel() == 0) return {idxs, dists};  // knn.cu:327-329
  TORCH_CHECK(p2_in.size(0) == N && lengths1_in.numel() == N && lengths2_in.numel() == N,
              "batch sizes differ");
  TORCH_CHECK(p1_in.scalar_type() == p2_in.scalar_type(), "p1 and p2 dtypes differ");
  TORCH_CHECK(lengths1_in.scalar_type() == at::kLong && lengths2_in.scalar_type() == at::kLong,
              "lengths must be int64");
  const at::Tensor l1 = lengths1_in.contiguous(), l2 = lengths2_in.contiguous();
  if (p1_in.scalar_type() == at::kBFloat16) {
    // bfloat16 (the reference raises): matrix-core kernel where it applies,
    // otherwise the float kernels on the exactly widened values
    const int64_t wsb = tpo_knn_workspace_size(TPO_BF16, N, P1, P2, D, K, (int)norm);
    if (wsb > 0) {
      const at::Tensor p1 = aligned16(p1_in.contiguous()), p2 = aligned16(p2_in.contiguous());
      at::Tensor work = at::empty({wsb}, p1.options().dtype(at::kByte));
      check_rc(tpo_knn_fwd(TPO_BF16, p1.data_ptr(), p2.data_ptr(), l1.data_ptr<int64_t>(),
                           l2.data_ptr<int64_t>(), N, P1, P2, D, K, (int)norm, (int)version,
                           idxs.data_ptr<int64_t>(), dists.data_ptr(), nullptr,
                           work.data_ptr(), wsb, stream_of(p1)),
               "knn_forward");
      return {idxs, dists};
    }
    auto r = knn_forward_hip(p1_in.to(at::kFloat), p2_in.to(at::kFloat), lengths1_in,
                             lengths2_in, norm, K, version);
    return {std::get<0>(r), std::get<1>(r).to(at::kBFloat16)};
  }
  const at::Tensor p1 = p1_in.contiguous(), p2 = p2_in.contiguous();
  const int dt = dtype_code(p1, "knn_forward");
  const int64_t ws = K == 1 ? tpo_knn_rows_workspace_size(dt, N, P1, P2, D, K, (int)norm)
                            : tpo_knn_workspace_size(dt, N, P1, P2, D, K, (int)norm);
  at::Tensor work = at::empty({ws > 0 ? ws : 1}, p1.options().dtype(at::kByte));
  check_rc(tpo_knn_fwd(dt, p1.data_ptr(), p2.data_ptr(), l1.data_ptr<int64_t>(),
                       l2.data_ptr<int64_t>(), N, P1, P2, D, K, (int)norm, (int)version,
                       idxs.data_ptr<int64_t>(), dists.data_ptr(), nullptr, work.data_ptr(), ws,
                       stream_of(p1)),
           "knn_forward");
  return {idxs, dists};
}

// knn_points(return_sorted=True) in one launch: the forward with each row
// sorted as the module's torch sort leaves it (knn/__init__.py:111-131).
// 2 <= K <= 32; the module keeps its own sort otherwise.
std::tuple<at::Tensor, at::Tensor> knn_forward_sorted_hip(const at::Tensor& p1_in,
                                                          const at::Tensor& p2_in,
                                                          const at::Tensor& lengths1_in,
                                                          const at::Tensor& lengths2_in,
                                                          int64_t norm, int64_t K,
                                                          int64_t version) {
  TORCH_CHECK(p1_in.device() == p2_in.device(), "p1 and p2 must be on the same device");
  TORCH_CHECK(p1_in.device() == lengths1_in.device(),
              "p1 and lengths1 must be on the same device");
  TORCH_CHECK(p1_in.device() == lengths2_in.device(),
              "p1 and lengths2 must be on the same device");
  check_hip(p1_in, "p1");
  c10::OptionalDeviceGuard guard(p1_in.device());
  TORCH_CHECK(p1_in.dim() == 3 && p2_in.dim() == 3, "knn_forward_sorted expects (N,P,D) tensors");
  const int64_t N = p1_in.size(0), P1 = p1_in.size(1), P2 = p2_in.size(1), D = p1_in.size(2);
  TORCH_CHECK((norm == 1) || (norm == 2), "Norm must be 1 or 2.");
  TORCH_CHECK(p2_in.size(2) == D, "Point sets must have the same last dimension");
  TORCH_CHECK(K >= 2 && K <= 32, "knn_forward_sorted needs 2 <= K <= 32");
  auto idxs = at::empty({N, P1, K}, lengths1_in.options().dtype(at::kLong));
  auto dists = at::empty({N, P1, K}, p1_in.options());
  if (idxs.numel() == 0) return {idxs, dists};
  TORCH_CHECK(p2_in.size(0) == N && lengths1_in.numel() == N && lengths2_in.numel() == N,
              "batch sizes differ");
  TORCH_CHECK(p1_in.scalar_type() == p2_in.scalar_type(), "p1 and p2 dtypes differ");
  TORCH_CHECK(lengths1_in.scalar_type() == at::kLong && lengths2_in.scalar_type() == at::kLong,
              "lengths must be int64");
  const at::Tensor l1 = lengths1_in.contiguous(), l2 = lengths2_in.contiguous();
  if (p1_in.scalar_type() == at::kBFloat16) {  // the forward's rows, then the sort in place
    std::tie(idxs, dists) = knn_forward_hip(p1_in, p2_in, lengths1_in, lengths2_in, norm, K, version);
    check_rc(tpo_knn_sort_rows(TPO_BF16, l2.data_ptr<int64_t>(), N, P1, K,
                               idxs.data_ptr<int64_t>(), dists.data_ptr(), stream_of(p1_in)),
             "knn_forward_sorted");
    return {idxs, dists};
  }
  const at::Tensor p1 = p1_in.contiguous(), p2 = p2_in.contiguous();
  const int dt = dtype_code(p1, "knn_forward_sorted");
  const int64_t ws = tpo_knn_rows_workspace_size(dt, N, P1, P2, D, K, (int)norm);
  at::Tensor work = at::empty({ws > 0 ? ws : 1}, p1.options().dtype(at::kByte));
  check_rc(tpo_knn_fwd_sorted(dt, p1.data_ptr(), p2.data_ptr(), l1.data_ptr<int64_t>(),
                              l2.data_ptr<int64_t>(), N, P1, P2, D, K, (int)norm, (int)version,
                              idxs.data_ptr<int64_t>(), dists.data_ptr(), nullptr,
                              work.data_ptr(), ws, stream_of(p1)),
           "knn_forward_sorted");
  return {idxs, dists};
}

// knn_gather's expand + gather + mask (knn/__init__.py:136-183) in one launch
at::Tensor knn_gather_hip(const at::Tensor& x_in, const at::Tensor& idx_in,
                          const at::Tensor& lengths_in) {
  check_hip(x_in, "x");
  c10::OptionalDeviceGuard guard(x_in.device());
  TORCH_CHECK(x_in.dim() == 3 && idx_in.dim() == 3, "knn_gather expects (N,M,U) and (N,L,K)");
  const int64_t N = x_in.size(0), M = x_in.size(1), U = x_in.size(2);
  const int64_t L = idx_in.size(1), K = idx_in.size(2);
  TORCH_CHECK(idx_in.size(0) == N, "x and idx must have same batch dimension.");
  TORCH_CHECK(idx_in.scalar_type() == at::kLong && lengths_in.scalar_type() == at::kLong,
              "idx and lengths must be int64");
  TORCH_CHECK(lengths_in.numel() == N, "lengths must have one entry per cloud");
  TORCH_CHECK(x_in.device() == idx_in.device() && x_in.device() == lengths_in.device(),
              "x, idx and lengths must be on the same device");
  const at::Tensor x = x_in.contiguous(), idx = idx_in.contiguous();
  const at::Tensor lengths = lengths_in.contiguous();
  at::Tensor out = at::empty({N, L, K, U}, x.options());
  int dt;
  switch (x.scalar_type()) {
    case at::kFloat: dt = TPO_F32; break;
    case at::kDouble: dt = TPO_F64; break;
    case at::kHalf: dt = TPO_F16; break;
    case at::kBFloat16: dt = TPO_BF16; break;
    default: TORCH_CHECK(false, "knn_gather not implemented for '", x.scalar_type(), "'");
  }
  TORCH_CHECK(M > 0 || out.numel() == 0, "knn_gather: x has no points");
  check_rc(tpo_knn_gather(dt, x.data_ptr(), idx.data_ptr<int64_t>(),
                          lengths.data_ptr<int64_t>(), N, M, L, K, U, out.data_ptr(),
                          stream_of(x)),
           "knn_gather");
  return out;
}

// knn_gather's gradient in x: records grouped by row and summed in LDS where
// the rows are short (tpo_knn_gather_bwd), torch's scatter otherwise.
at::Tensor knn_gather_backward_hip(const at::Tensor& go_in, const at::Tensor& idx_in,
                                   const at::Tensor& lengths_in, int64_t M) {
  check_hip(go_in, "grad_out");
  c10::OptionalDeviceGuard guard(go_in.device());
  TORCH_CHECK(go_in.dim() == 4 && idx_in.dim() == 3,
              "knn_gather_backward expects (N,L,K,U) and (N,L,K)");
  const int64_t N = go_in.size(0), L = go_in.size(1), K = go_in.size(2), U = go_in.size(3);
  TORCH_CHECK(idx_in.size(0) == N && idx_in.size(1) == L && idx_in.size(2) == K,
              "idx shape differs from grad_out");
  TORCH_CHECK(idx_in.scalar_type() == at::kLong && lengths_in.scalar_type() == at::kLong,
              "idx and lengths must be int64");
  TORCH_CHECK(lengths_in.numel() == N, "lengths must have one entry per cloud");
  TORCH_CHECK(go_in.device() == idx_in.device() && go_in.device() == lengths_in.device(),
              "grad_out, idx and lengths must be on the same device");
  TORCH_CHECK(M >= 0, "M must be non-negative");
  const at::Tensor go = go_in.contiguous(), idx = idx_in.contiguous();
  const at::Tensor lengths = lengths_in.contiguous();
  int dt = -1;
  if (go.scalar_type() == at::kFloat) dt = TPO_F32;
  if (go.scalar_type() == at::kDouble) dt = TPO_F64;
  if (go.scalar_type() == at::kHalf) dt = TPO_F16;
  const int64_t wsb = dt < 0 ? 0 : tpo_knn_gather_bwd_workspace_size(dt, N, M, L, K, U);
  if (wsb > 0) {
    at::Tensor gx = at::empty({N, M, U}, go.options());
    at::Tensor ws = at::empty({wsb}, go.options().dtype(at::kByte));
    check_rc(tpo_knn_gather_bwd(dt, go.data_ptr(), idx.data_ptr<int64_t>(),
                                lengths.data_ptr<int64_t>(), N, M, L, K, U, gx.data_ptr(),
                                ws.data_ptr(), wsb, stream_of(go)),
             "knn_gather_backward");
    return gx;
  }
  at::Tensor gx = at::zeros({N, M, U}, go.options());
  if (go.numel() == 0 || gx.numel() == 0) return gx;
  const at::Tensor keep = at::arange(K, idx.options()).unsqueeze(0).lt(lengths.view({N, 1}));
  const at::Tensor g = at::where(keep.view({N, 1, K, 1}), go, at::zeros({}, go.options()));
  const at::Tensor j = idx.clamp(0, M - 1).view({N, L * K, 1}).expand({N, L * K, U});
  return gx.scatter_add_(1, j, g.reshape({N, L * K, U}));
}

std::tuple<at::Tensor, at::Tensor> knn_backward_hip(const at::Tensor& p1_in,
                                                    const at::Tensor& p2_in,
                                                    const at::Tensor& lengths1_in,
                                                    const at::Tensor& lengths2_in,
                                                    const at::Tensor& idxs_in, int64_t norm,
                                                    const at::Tensor& grad_dists_in) {
  check_hip(p1_in, "p1");
  c10::OptionalDeviceGuard guard(p1_in.device());
  const int64_t N = p1_in.size(0), P1 = p1_in.size(1), P2 = p2_in.size(1), D = p1_in.size(2);
  const int64_t K = idxs_in.size(2);
  // knn.cu:487-492
  TORCH_CHECK(p2_in.size(2) == D, "Point sets must have the same last dimension");
  TORCH_CHECK(idxs_in.size(0) == N, "KNN idxs must have the same batch dimension");
  TORCH_CHECK(idxs_in.size(1) == P1, "KNN idxs must have the same point dimension as p1");
  TORCH_CHECK(grad_dists_in.size(0) == N);
  TORCH_CHECK(grad_dists_in.size(1) == P1);
  TORCH_CHECK(grad_dists_in.size(2) == K);
  TORCH_CHECK((norm == 1) || (norm == 2), "Norm must be 1 or 2.");
  auto g1 = at::empty_like(p1_in, at::MemoryFormat::Contiguous);
  auto g2 = at::empty_like(p2_in, at::MemoryFormat::Contiguous);
  if (g1.numel() == 0 || g2.numel() == 0) {  // knn.cu:497-499
    g1.zero_();
    g2.zero_();
    return {g1, g2};
  }
  if (p1_in.scalar_type() == at::kBFloat16) {  // computed in float, rounded once
    auto r = knn_backward_hip(p1_in.to(at::kFloat), p2_in.to(at::kFloat), lengths1_in,
                              lengths2_in, idxs_in, norm, grad_dists_in.to(at::kFloat));
    return {std::get<0>(r).to(at::kBFloat16), std::get<1>(r).to(at::kBFloat16)};
  }
  const at::Tensor p1 = p1_in.contiguous(), p2 = p2_in.contiguous();
  const at::Tensor l1 = lengths1_in.contiguous(), l2 = lengths2_in.contiguous();
  const at::Tensor idxs = idxs_in.contiguous();
  const at::Tensor gd = grad_dists_in.to(p1.scalar_type()).contiguous();
  const int dt = dtype_code(p1, "knn_backward");
  // grad_p2 without global atomics: the entry terms are grouped by reference
  // rows in the workspace (tpo_knn_bwd_ws)
  const int64_t wsb = tpo_knn_bwd_workspace_size(dt, N, P1, P2, D, K);
  at::Tensor ws;
  if (wsb > 0) ws = at::empty({wsb}, p1.options().dtype(at::kByte));
  check_rc(tpo_knn_bwd_ws(dt, p1.data_ptr(), p2.data_ptr(), l1.data_ptr<int64_t>(),
                          l2.data_ptr<int64_t>(), idxs.data_ptr<int64_t>(), (int)norm,
                          gd.data_ptr(), N, P1, P2, D, K, g1.data_ptr(), g2.data_ptr(),
                          wsb > 0 ? ws.data_ptr() : nullptr, wsb, stream_of(p1)),
           "knn_backward");
  return {g1, g2};
}

// Autograd of the KNN operators in C++, as the Chamfer loss's: a step's forward
// and backward run no Python.  Gradients of outputs that a loss leaves out are
// not materialised; the index outputs carry none (knn/__init__.py:6-28).
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

template <typename Op>
auto typed_op(const char* name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Op>();
}

template <bool SORTED>
auto knn_op() {
  static auto op = typed_op<std::tuple<at::Tensor, at::Tensor>(
      const at::Tensor&, const at::Tensor&, const at::Tensor&, const at::Tensor&, int64_t, int64_t,
      int64_t)>(SORTED ? "torch_point_ops_knn::knn_forward_sorted"
                       : "torch_point_ops_knn::knn_forward");
  return op;
}
auto knn_gather_op() {
  static auto op = typed_op<at::Tensor(const at::Tensor&, const at::Tensor&, const at::Tensor&)>(
      "torch_point_ops_knn::knn_gather");
  return op;
}
auto gather_points_op() {
  static auto op = typed_op<at::Tensor(const at::Tensor&, const at::Tensor&)>(
      "torch_point_ops_fps::gather_points_forward");
  return op;
}

template <bool SORTED>
class KnnFunction : public torch::autograd::Function<KnnFunction<SORTED>> {
 public:
  static variable_list forward(AutogradContext* ctx, const at::Tensor& p1, const at::Tensor& p2,
                               const at::Tensor& lengths1, const at::Tensor& lengths2,
                               int64_t norm, int64_t K, int64_t version) {
    at::Tensor idxs, dists;
    {
      at::AutoDispatchBelowADInplaceOrView below;
      std::tie(idxs, dists) = knn_op<SORTED>().call(p1, p2, lengths1, lengths2, norm, K, version);
    }
    ctx->save_for_backward({p1, p2, lengths1, lengths2, idxs});
    ctx->saved_data["norm"] = norm;
    ctx->mark_non_differentiable({idxs});
    ctx->set_materialize_grads(false);
    return {idxs, dists};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    static auto op = typed_op<std::tuple<at::Tensor, at::Tensor>(
        const at::Tensor&, const at::Tensor&, const at::Tensor&, const at::Tensor&,
        const at::Tensor&, int64_t, const at::Tensor&)>("torch_point_ops_knn::knn_backward");
    at::Tensor g1, g2, none;
    if (grads[1].defined()) {
      const auto s = ctx->get_saved_variables();
      std::tie(g1, g2) =
          op.call(s[0], s[1], s[2], s[3], s[4], ctx->saved_data["norm"].toInt(), grads[1]);
    }
    return {g1, g2, none, none, none, none, none};
  }
};

template <bool SORTED>
std::tuple<at::Tensor, at::Tensor> knn_forward_autograd(
    const at::Tensor& p1, const at::Tensor& p2, const at::Tensor& lengths1,
    const at::Tensor& lengths2, int64_t norm, int64_t K, int64_t version) {
  if (!followed(p1) && !followed(p2)) {
    at::AutoDispatchBelowADInplaceOrView below;
    return knn_op<SORTED>().call(p1, p2, lengths1, lengths2, norm, K, version);
  }
  auto out = KnnFunction<SORTED>::apply(p1, p2, lengths1, lengths2, norm, K, version);
  return {out[0], out[1]};
}

class KnnGatherFunction : public torch::autograd::Function<KnnGatherFunction> {
 public:
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& x, const at::Tensor& idx,
                            const at::Tensor& lengths) {
    ctx->save_for_backward({idx, lengths});
    ctx->saved_data["M"] = x.sym_size(1);  // symbolic while a program is traced
    at::AutoDispatchBelowADInplaceOrView below;
    return knn_gather_op().call(x, idx, lengths);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    static auto op =
        typed_op<at::Tensor(const at::Tensor&, const at::Tensor&, const at::Tensor&, c10::SymInt)>(
            "torch_point_ops_knn::knn_gather_backward");
    const auto s = ctx->get_saved_variables();
    const c10::SymInt M = ctx->saved_data["M"].toSymInt();
    if (at::GradMode::is_enabled())  // its own gradient is the gather (knn/__init__.py)
      return {op.call(grads[0], s[0], s[1], M), at::Tensor(), at::Tensor()};
    at::AutoDispatchBelowADInplaceOrView below;
    return {op.call(grads[0], s[0], s[1], M), at::Tensor(), at::Tensor()};
  }
};

at::Tensor knn_gather_autograd(const at::Tensor& x, const at::Tensor& idx,
                               const at::Tensor& lengths) {
  TORCH_CHECK(x.dim() == 3, "knn_gather expects (N,M,U) and (N,L,K)");
  if (!followed(x)) {
    at::AutoDispatchBelowADInplaceOrView below;
    return knn_gather_op().call(x, idx, lengths);
  }
  return KnnGatherFunction::apply(x, idx, lengths);
}

// ---------------------------------------------------------------------- fps
at::Tensor fps_forward_hip(const at::Tensor& points_in, int64_t nsamples) {
  check_hip(points_in, "points");
  c10::OptionalDeviceGuard guard(points_in.device());
  TORCH_CHECK(points_in.dim() == 3, "fps_forward expects (N,P,3)");
  const int64_t B = points_in.size(0), P = points_in.size(1), D = points_in.size(2);
  // fps.cu:282-284
  TORCH_CHECK(D == 3, "FPS only supports 3D points, but got dimension ", D);
  TORCH_CHECK(nsamples > 0, "nsamples must be positive, but got ", nsamples);
  TORCH_CHECK(nsamples <= P, "nsamples (", nsamples, ") cannot exceed number of points (", P,
              ")");
  auto idx = at::empty({B, nsamples}, points_in.options().dtype(at::kLong));
  if (idx.numel() == 0) return idx;
  const at::Tensor points = points_in.contiguous();
  const int dt = dtype_code(points, "fps_forward");
  const int64_t ws = tpo_fps_workspace_size(dt, B, P);
  TORCH_CHECK(ws >= 0, "fps_forward: ", tpo_last_error());
  at::Tensor work = at::empty({ws > 0 ? ws : 1}, points.options().dtype(at::kByte));
  check_rc(tpo_fps_fwd(dt, points.data_ptr(), B, P, nsamples, idx.data_ptr<int64_t>(),
                       work.data_ptr(), ws, stream_of(points)),
           "fps_forward");
  return idx;
}

// fps.cpp:144-155 checks; served by the exact FPS kernel (kd_depth only
// validated), which the reference's tests require to agree with FPS.
at::Tensor quick_fps_forward_hip(const at::Tensor& points, int64_t nsamples, int64_t kd_depth) {
  TORCH_CHECK(points.dim() == 3 && points.size(2) == 3,
              "Quick FPS only supports 3D points, but got dimension ",
              points.dim() == 3 ? points.size(2) : -1);
  TORCH_CHECK(kd_depth > 0 && kd_depth <= 10, "kd_depth must be between 1 and 10, but got ",
              kd_depth);
  return fps_forward_hip(points, nsamples);
}

at::Tensor gather_points_forward_hip(const at::Tensor& points_in, const at::Tensor& idx_in) {
  TORCH_CHECK(points_in.device() == idx_in.device(),
              "points and idx must be on the same device");  // fps.cu:321
  check_hip(points_in, "points");
  c10::OptionalDeviceGuard guard(points_in.device());
  TORCH_CHECK(points_in.dim() == 3 && idx_in.dim() == 2, "gather_points expects (N,C,P), (N,M)");
  TORCH_CHECK(idx_in.scalar_type() == at::kLong, "gather_points expects int64 indices");
  const int64_t B = points_in.size(0), C = points_in.size(1), P = points_in.size(2);
  const int64_t M = idx_in.size(1);
  TORCH_CHECK(idx_in.size(0) == B, "batch sizes differ");
  auto out = at::empty({B, C, M}, points_in.options());
  if (out.numel() == 0) return out;
  const at::Tensor points = points_in.contiguous(), idx = idx_in.contiguous();
  const int dt = dtype_code(points, "gather_points_forward");
  check_rc(tpo_gather_fwd(dt, points.data_ptr(), idx.data_ptr<int64_t>(), B, C, P, M,
                          out.data_ptr(), stream_of(points)),
           "gather_points_forward");
  return out;
}

at::Tensor gather_points_backward_hip(const at::Tensor& grad_in, const at::Tensor& idx_in,
                                      int64_t n) {
  TORCH_CHECK(grad_in.device() == idx_in.device(),
              "grad_out and idx must be on the same device");  // fps.cu:367
  check_hip(grad_in, "grad_out");
  c10::OptionalDeviceGuard guard(grad_in.device());
  TORCH_CHECK(grad_in.dim() == 3 && idx_in.dim() == 2, "gather_points_backward expects 3D/2D");
  TORCH_CHECK(idx_in.scalar_type() == at::kLong, "gather_points expects int64 indices");
  const int64_t B = grad_in.size(0), C = grad_in.size(1), M = grad_in.size(2);
  TORCH_CHECK(n >= 0, "n must be non-negative");
  auto out = at::empty({B, C, n}, grad_in.options());
  if (out.numel() == 0) return out;
  const at::Tensor go = grad_in.contiguous(), idx = idx_in.contiguous();
  TORCH_CHECK(idx.size(0) == B && idx.size(1) == M, "idx shape differs from grad_out");
  const int dt = dtype_code(go, "gather_points_backward");
  const int64_t ws = tpo_gather_bwd_workspace_size(B, n);
  at::Tensor work = at::empty({ws > 0 ? ws : 1}, go.options().dtype(at::kByte));
  check_rc(tpo_gather_bwd(dt, go.data_ptr(), idx.data_ptr<int64_t>(), B, C, n, M, out.data_ptr(),
                          work.data_ptr(), ws, stream_of(go)),
           "gather_points_backward");
  return out;
}

// gather_points' autograd (fps/__init__.py:8-30) in C++
class GatherPointsFunction : public torch::autograd::Function<GatherPointsFunction> {
 public:
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& points, const at::Tensor& idx) {
    ctx->save_for_backward({idx});
    ctx->saved_data["n"] = points.sym_size(2);  // symbolic while a program is traced
    at::AutoDispatchBelowADInplaceOrView below;
    return gather_points_op().call(points, idx);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    static auto op = typed_op<at::Tensor(const at::Tensor&, const at::Tensor&, int64_t)>(
        "torch_point_ops_fps::gather_points_backward");
    const auto s = ctx->get_saved_variables();
    const int64_t n = ctx->saved_data["n"].toSymInt().guard_int(__FILE__, __LINE__);  // the schema's int
    return {op.call(grads[0], s[0], n), at::Tensor()};
  }
};

at::Tensor gather_points_autograd(const at::Tensor& points, const at::Tensor& idx) {
  TORCH_CHECK(points.dim() == 3, "gather_points expects (N,C,P), (N,M)");
  if (!followed(points)) {
    at::AutoDispatchBelowADInplaceOrView below;
    return gather_points_op().call(points, idx);
  }
  return GatherPointsFunction::apply(points, idx);
}

// ---------------------------------------------------------------------- emd
// emd.cu:11-13: CHECK_CUDA + CHECK_CONTIGUOUS
void check_emd_input(const at::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

std::tuple<at::Tensor, at::Tensor> emd_forward_hip(const at::Tensor& xyz1,
                                                   const at::Tensor& xyz2) {
  check_emd_input(xyz1, "xyz1");
  check_emd_input(xyz2, "xyz2");
  // emd.cu:309-311
  TORCH_CHECK(xyz1.dim() == 3 && xyz2.dim() == 3, "Input tensors must be 3D");
  TORCH_CHECK(xyz1.size(0) == xyz2.size(0), "Input tensors must have the same batch size");
  TORCH_CHECK(xyz1.size(2) == 3 && xyz2.size(2) == 3, "Input tensors must have 3 channels");
  TORCH_CHECK(xyz1.scalar_type() == xyz2.scalar_type(), "dtypes differ");
  TORCH_CHECK(xyz1.device() == xyz2.device(), "xyz1 and xyz2 must be on the same device");
  c10::OptionalDeviceGuard guard(xyz1.device());
  const int64_t B = xyz1.size(0), n = xyz1.size(1), m = xyz2.size(1);
  const int dt = dtype_code(xyz1, "emd_forward");
  at::Tensor cost = at::empty({B}, xyz1.options());
  at::Tensor match = at::empty({B, m, n}, xyz1.options());
  const int64_t ws_bytes = tpo_emd_workspace_size(dt, B, n, m);
  TORCH_CHECK(ws_bytes >= 0, "emd_forward: ", tpo_last_error());
  at::Tensor ws;
  if (ws_bytes > 0) ws = at::empty({ws_bytes}, xyz1.options().dtype(at::kByte));
  check_rc(tpo_emd_fwd(dt, xyz1.data_ptr(), xyz2.data_ptr(), B, n, m, cost.data_ptr(),
                       match.data_ptr(), ws_bytes > 0 ? ws.data_ptr() : nullptr, ws_bytes,
                       stream_of(xyz1)),
           "emd_forward");
  return {cost, match};
}

std::tuple<at::Tensor, at::Tensor> emd_backward_hip(const at::Tensor& grad_cost_in,
                                                    const at::Tensor& xyz1, const at::Tensor& xyz2,
                                                    const at::Tensor& match) {
  TORCH_CHECK(grad_cost_in.is_cuda(), "grad_cost must be a CUDA tensor");
  check_emd_input(xyz1, "xyz1");
  check_emd_input(xyz2, "xyz2");
  check_emd_input(match, "match");
  TORCH_CHECK(xyz1.dim() == 3 && xyz2.dim() == 3, "Input tensors must be 3D");
  c10::OptionalDeviceGuard guard(xyz1.device());
  const int64_t B = xyz1.size(0), n = xyz1.size(1), m = xyz2.size(1);
  TORCH_CHECK(xyz2.size(0) == B && grad_cost_in.numel() == B, "batch sizes differ");
  TORCH_CHECK(match.scalar_type() == xyz1.scalar_type() && xyz2.scalar_type() == xyz1.scalar_type(),
              "dtypes differ");
  TORCH_CHECK(match.numel() == B * m * n, "match must be (B, m, n)");
  const int dt = dtype_code(xyz1, "emd_backward");
  const at::Tensor grad_cost = grad_cost_in.to(xyz1.scalar_type()).contiguous();
  at::Tensor g1 = at::empty_like(xyz1), g2 = at::empty_like(xyz2);
  const int64_t ws_bytes = tpo_emd_workspace_size(dt, B, n, m);
  TORCH_CHECK(ws_bytes >= 0, "emd_backward: ", tpo_last_error());
  at::Tensor ws;
  if (ws_bytes > 0) ws = at::empty({ws_bytes}, xyz1.options().dtype(at::kByte));
  check_rc(tpo_emd_bwd(dt, grad_cost.data_ptr(), xyz1.data_ptr(), xyz2.data_ptr(), match.data_ptr(),
                       B, n, m, g1.data_ptr(), g2.data_ptr(), ws_bytes > 0 ? ws.data_ptr() : nullptr,
                       ws_bytes, stream_of(xyz1)),
           "emd_backward");
  return {g1, g2};
}

// emd.cpp:19-28
std::tuple<at::Tensor, at::Tensor> emd_forward_cpu(const at::Tensor&, const at::Tensor&) {
  TORCH_CHECK(false, "emd_forward is not implemented for CPU");
}
std::tuple<at::Tensor, at::Tensor> emd_backward_cpu(const at::Tensor&, const at::Tensor&,
                                                    const at::Tensor&, const at::Tensor&) {
  TORCH_CHECK(false, "emd_backward is not implemented for CPU");
}

}  // namespace

TORCH_LIBRARY(torch_point_ops_chamfer, m) {
  m.def("chamfer_forward(Tensor xyz1, Tensor xyz2) -> (Tensor, Tensor, Tensor, Tensor)");
  m.def("chamfer_backward(Tensor xyz1, Tensor xyz2, Tensor idx1, Tensor idx2, "
        "Tensor grad_dist1, Tensor grad_dist2) -> (Tensor, Tensor)");
  // the module's reduction fused into the kernels (no reference schema)
  m.def("chamfer_loss_forward(Tensor xyz1, Tensor xyz2, bool mean) -> (Tensor, Tensor, Tensor)");
  m.def("chamfer_loss_backward(Tensor xyz1, Tensor xyz2, Tensor idx1, Tensor idx2, "
        "Tensor grad_loss, bool mean) -> (Tensor, Tensor)");
}
TORCH_LIBRARY_IMPL(torch_point_ops_chamfer, CPU, m) {
  m.impl("chamfer_forward", &chamfer_forward_cpu);
  m.impl("chamfer_backward", &chamfer_backward_cpu);
  m.impl("chamfer_loss_forward", &chamfer_loss_forward_cpu);
  m.impl("chamfer_loss_backward", &chamfer_loss_backward_cpu);
}
TORCH_LIBRARY_IMPL(torch_point_ops_chamfer, Autograd, m) {
  m.impl("chamfer_forward", &chamfer_forward_autograd);
  m.impl("chamfer_loss_forward", &chamfer_loss_forward_autograd);
}
TORCH_LIBRARY_IMPL(torch_point_ops_chamfer, CUDA, m) {
  m.impl("chamfer_forward", &chamfer_forward_hip);
  m.impl("chamfer_backward", &chamfer_backward_hip);
  m.impl("chamfer_loss_forward", &chamfer_loss_forward_hip);
  m.impl("chamfer_loss_backward", &chamfer_loss_backward_hip);
}

TORCH_LIBRARY(torch_point_ops_knn, m) {
  m.def("knn_forward(Tensor p1, Tensor p2, Tensor lengths1, Tensor lengths2, "
        "int norm, int K, int version) -> (Tensor, Tensor)");
  m.def("knn_backward(Tensor p1, Tensor p2, Tensor lengths1, Tensor lengths2, "
        "Tensor idxs, int norm, Tensor grad_dists) -> (Tensor, Tensor)");
  // the forward and knn_points' sort in one launch (no reference schema)
  m.def("knn_forward_sorted(Tensor p1, Tensor p2, Tensor lengths1, Tensor lengths2, "
        "int norm, int K, int version) -> (Tensor, Tensor)");
  m.def("knn_gather(Tensor x, Tensor idx, Tensor lengths) -> Tensor");
  m.def("knn_gather_backward(Tensor grad_out, Tensor idx, Tensor lengths, SymInt M) -> Tensor");
}
TORCH_LIBRARY_IMPL(torch_point_ops_knn, CUDA, m) {
  m.impl("knn_forward", &knn_forward_hip);
  m.impl("knn_forward_sorted", &knn_forward_sorted_hip);
  m.impl("knn_gather", &knn_gather_hip);
  m.impl("knn_gather_backward", &knn_gather_backward_hip);
  m.impl("knn_backward", &knn_backward_hip);
}

TORCH_LIBRARY_IMPL(torch_point_ops_knn, Autograd, m) {
  m.impl("knn_forward", &knn_forward_autograd<false>);
  m.impl("knn_forward_sorted", &knn_forward_autograd<true>);
  m.impl("knn_gather", &knn_gather_autograd);
}

TORCH_LIBRARY(torch_point_ops_fps, m) {
  m.def("fps_forward(Tensor points, int nsamples) -> Tensor");
  m.def("gather_points_forward(Tensor points, Tensor idx) -> Tensor");
  m.def("gather_points_backward(Tensor grad_out, Tensor idx, int n) -> Tensor");
}
TORCH_LIBRARY_IMPL(torch_point_ops_fps, CUDA, m) {
  m.impl("fps_forward", &fps_forward_hip);
  m.impl("gather_points_forward", &gather_points_forward_hip);
  m.impl("gather_points_backward", &gather_points_backward_hip);
}

TORCH_LIBRARY_IMPL(torch_point_ops_fps, Autograd, m) {
  m.impl("gather_points_forward", &gather_points_autograd);
}

TORCH_LIBRARY(torch_point_ops_quick_fps, m) {
  m.def("quick_fps_forward(Tensor points, int nsamples, int kd_depth=4) -> Tensor");
}
TORCH_LIBRARY_IMPL(torch_point_ops_quick_fps, CUDA, m) {
  m.impl("quick_fps_forward", &quick_fps_forward_hip);
}

TORCH_LIBRARY(torch_point_ops_emd, m) {
  m.def("emd_forward(Tensor xyz1, Tensor xyz2) -> (Tensor, Tensor)");
  m.def("emd_backward(Tensor grad_cost, Tensor xyz1, Tensor xyz2, Tensor match) -> (Tensor, Tensor)");
}
TORCH_LIBRARY_IMPL(torch_point_ops_emd, CPU, m) {
  m.impl("emd_forward", &emd_forward_cpu);
  m.impl("emd_backward", &emd_backward_cpu);
}
TORCH_LIBRARY_IMPL(torch_point_ops_emd, CUDA, m) {
  m.impl("emd_forward", &emd_forward_hip);
  m.impl("emd_backward", &emd_backward_hip);
}

}  // namespace torch_point_ops

// Importing torch_point_ops._C loads this library, whose static
// initialisers above register the operators (the reference's pattern,
// chamfer.cpp:46-63).
extern "C" PyObject* PyInit__C(void) {
  static struct PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_C", nullptr, -1, nullptr};
  return PyModule_Create(&module_def);
}
