// FP32 instances of the vector-ALU forms (kernels_valu.hpp).
#include "kernels_valu.hpp"

namespace fmca_amd {
template hipError_t launch_valu<float>(bool, const ValuLaunch<float> &);
}
