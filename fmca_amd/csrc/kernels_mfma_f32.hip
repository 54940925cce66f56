// FP32 instances of the matrix-core forms (kernels_mfma.hpp) and the leaf
// moments.
#include "kernels_mfma.hpp"

namespace fmca_amd {

// Leaf moments of the FP32 forms on the matrix cores (q <= 128, >= 8 rhs);
// false: the caller takes the VALU kernel.
bool upward_leaf_mfma_supported(int D, int P1, int q, int nrhs) {
  return q <= 128 && nrhs >= kMfmaMinRhs && D >= 1 && D <= 3 &&
         ((size_t)D * P1 * 68 + 64 * 36) * sizeof(float) <= 64 * 1024;
}

hipError_t launch_upward_leaf_mfma(const DevTreeView<float> &tr, const InterpParams<float> &ip,
                                   const float *xs, int nrhs, float *mom, hipStream_t stream) {
  const int D = tr.dim, P1 = ip.P1;
  const int NT = nrhs > 16 ? 2 : 1;
  const size_t lds = ((size_t)D * P1 * 68 + (size_t)64 * (16 * NT + 4)) * sizeof(float);
#define FMCA_UPL(DV, NTV)                                                                   \
  hipLaunchKernelGGL((k_upward_leaf_mfma<DV, NTV>), dim3(tr.nleaves), dim3(256), lds, stream, \
                     tr, ip, xs, nrhs, mom)
  if (D == 1) {
    if (NT == 2) FMCA_UPL(1, 2); else FMCA_UPL(1, 1);
  } else if (D == 2) {
    if (NT == 2) FMCA_UPL(2, 2); else FMCA_UPL(2, 1);
  } else {
    if (NT == 2) FMCA_UPL(3, 2); else FMCA_UPL(3, 1);
  }
#undef FMCA_UPL
  return hipGetLastError();
}

template bool mfma_supported<float>(bool, int, int, int, int, int, int, int);
template hipError_t launch_mfma<float>(bool, const MfmaLaunch<float> &);

}  // namespace fmca_amd
