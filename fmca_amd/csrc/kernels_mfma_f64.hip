// FP64 instances of the matrix-core forms (kernels_mfma.hpp).
#include "kernels_mfma.hpp"

namespace fmca_amd {

template bool mfma_supported<double>(bool, int, int, int, int, int, int, int);
template hipError_t launch_mfma<double>(bool, const MfmaLaunch<double> &);

}  // namespace fmca_amd
