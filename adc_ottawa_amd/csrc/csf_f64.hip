// FP64 instantiations of the CSF-form virtual contractions.
#include "csf_virt.hpp"

namespace adc2g {

template void launch_csf_down<double>(const CsfGeo&, const CsfPlan&, const double*, const double*, const double*,
                                   const double*, double*, hipStream_t);
template void launch_csf_up<double>(const CsfGeo&, const CsfPlan&, const double*, const double*, const double*, double*,
                                 hipStream_t);

template void launch_csf_thin<double>(const CsfGeo&, const CsfPlan&, const double*, const double*, const double*,
                                   const double*, double*, double*, hipStream_t);

}  // namespace adc2g
