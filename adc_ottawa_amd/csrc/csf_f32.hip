// FP32 instantiations of the CSF-form virtual contractions.
#include "csf_virt.hpp"

namespace adc2g {

template void launch_csf_down<float>(const CsfGeo&, const CsfPlan&, const double*, const double*, const double*,
                                   const float*, float*, hipStream_t);
template void launch_csf_up<float>(const CsfGeo&, const CsfPlan&, const double*, const double*, const float*, double*,
                                 hipStream_t);

template void launch_csf_thin<float>(const CsfGeo&, const CsfPlan&, const double*, const double*, const double*,
                                   const float*, double*, float*, hipStream_t);

}  // namespace adc2g
