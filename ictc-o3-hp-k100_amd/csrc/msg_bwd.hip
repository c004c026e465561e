// CSR graph message first-adjoint launchers: receiver-owned gate / harmonic
// gradients, then the source-owned feature gradient.
#include "ictc_launch.h"

namespace ictc {

namespace {
struct MsgBwd {
  const Operands& a;
  const int64_t *src, *dst;
  Csr dcsr, scsr;
  const float* grad;
  float *dx, *dsh, *dg, *ws;
  hipStream_t st;
  template <class T, GateGrad GRAD>
  void src_pass(int G, int sum) {
    const dim3 grid(blocks_for((a.rows + 1) * sum), G);
    if (a.weight)
      hipLaunchKernelGGL((msg_bwd_src_kernel<T, GRAD, true>), grid, dim3(kBlock), 0, st, a, dst, scsr, grad, dx, dsh, ws,
                         dg, nullptr, nullptr, nullptr, sum);
    else
      hipLaunchKernelGGL((msg_bwd_src_kernel<T, GRAD, false>), grid, dim3(kBlock), 0, st, a, dst, scsr, grad, dx, dsh,
                         ws, dg, nullptr, nullptr, nullptr, sum);
  }
  template <class T>
  hipError_t run() {
    const int G = channel_groups(a.channels), sum = sum_parts(a.rows, G, kSourceSumWaves);
    // One source-owned pass for all three (rows + 1 slots: the last covers the out-of-range tail).
    if (dx && (dsh || dg)) {
      if (dg && a.dg_acc) src_pass<T, kAddGrad>(G, sum);
      else if (dg) src_pass<T, kStoreGrad>(G, sum);
      else src_pass<T, kNoGrad>(G, sum);
      hipError_t err = hipGetLastError();
      if (err != hipSuccess) return err;
      if (dsh) return launch_group_sum(dsh, ws, a.edges * T::NY, G - 1, st);
      return hipSuccess;
    }
    if (dsh || dg) {
      // rows + 1 row slots: the last one zero-fills the out-of-range tail segment.
      const int parts = row_parts(a.rows + 1, G);
      hipLaunchKernelGGL((msg_bwd_edge_kernel<T, false>), dim3(blocks_for((a.rows + 1) * parts), G), dim3(kBlock),
                         0, st, a, src, dcsr, grad, dsh, ws, dg, parts, nullptr, nullptr, nullptr);
      hipError_t err = hipGetLastError();
      if (err != hipSuccess) return err;
      if (dsh && (err = launch_group_sum(dsh, ws, a.edges * T::NY, G - 1, st)) != hipSuccess) return err;
    }
    if (dx) {
      hipLaunchKernelGGL((msg_bwd_x_kernel<T>), dim3(blocks_for(a.rows * sum), G), dim3(kBlock),
                         bwd_x_lds_cap<T>(a.rows), st, a, dst, scsr, grad, dx, sum);
      return hipGetLastError();
    }
    return hipSuccess;
  }
};
}  // namespace

hipError_t launch_msg_bwd(const TpShape& s, const Operands& a, const int64_t* src, const int64_t* dst, Csr dcsr,
                          Csr scsr, const float* grad, float* dx, float* dsh, float* dg, float* ws, hipStream_t st) {
  return dispatch_tp(s, MsgBwd{a, src, dst, dcsr, scsr, grad, dx, dsh, dg, ws, st});
}

}  // namespace ictc
