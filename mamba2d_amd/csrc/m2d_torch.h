// m2d_torch.h -- what the parts of the PyTorch shim share: the operators of m2d_torch.cpp as C++ functions.
#ifndef M2D_TORCH_H
#define M2D_TORCH_H
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/hip/HIPStream.h>

#include <tuple>
#include <vector>

#include "m2dscan.h"

namespace m2dshim {

using at::Tensor;

inline void check(int status) { TORCH_CHECK(status == M2D_OK, "m2dscan: ", m2d_status_str(status), " (status ", status, ")"); }
inline hipStream_t current_stream(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

std::tuple<Tensor, Tensor> scan_fwd(const Tensor& x, const Tensor& dT, const Tensor& dL, const Tensor& AT, const Tensor& AL,
                                    const Tensor& BT, const Tensor& BL, const Tensor& C, const Tensor& D, bool save_ckpt,
                                    bool flip, bool raw_params, bool packed_bc, int64_t ckpt_interval);
std::tuple<Tensor, Tensor> scan_y(const Tensor& x, const Tensor& dT, const Tensor& dL, const Tensor& AT, const Tensor& AL,
                                  const Tensor& BT, const Tensor& BL, const Tensor& C, const Tensor& D, bool save_ckpt,
                                  bool flip, bool raw_params, bool packed_bc, int64_t ckpt_interval);
std::vector<Tensor> scan_bwd(const Tensor& x, const Tensor& dT, const Tensor& dL, const Tensor& AT, const Tensor& AL,
                             const Tensor& BT, const Tensor& BL, const Tensor& C, const Tensor& D, const Tensor& dy,
                             const Tensor& ckpt, bool flip, bool raw_params, bool packed_bc, bool dpre, int64_t ckpt_interval,
                             bool sum_parts);
std::vector<Tensor> proj_fwd(const Tensor& x, const Tensor& Wx, const Tensor& wT, const Tensor& bT, const Tensor& wL,
                             const Tensor& bL, int64_t N, bool round_weights, bool packed_bc);
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> proj_bwd(const Tensor& x, const Tensor& low, const Tensor& dT, const Tensor& dL,
                                                            const Tensor& Wx, const Tensor& wT, const Tensor& wL, const Tensor& ddT,
                                                            const Tensor& ddL, const Tensor& dBT, const Tensor& dBL, const Tensor& dC,
                                                            Tensor dx, bool round_weights, bool dpre, int64_t sum_parts);

std::vector<Tensor> widen(at::TensorList in);      // m2d_infer.cpp

// Operator m2dscan::<name> through the dispatcher, for an autograd function whose backward is itself recorded
// (create_graph): the library has no second derivatives, and the dispatched operators are the ones that say so, with a
// warning, when somebody differentiates through them.
template <typename F>
c10::TypedOperatorHandle<F> dispatched(const char* name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<F>();
}

}  // namespace m2dshim
#endif
