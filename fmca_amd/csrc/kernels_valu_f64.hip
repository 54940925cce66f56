// FP64 instances of the vector-ALU forms (kernels_valu.hpp).
#include "kernels_valu.hpp"

namespace fmca_amd {
template hipError_t launch_valu<double>(bool, const ValuLaunch<double> &);
}
