// The mobility solve in FP32.
#include "fcm_run.hpp"

namespace fs {
template int FcmImpl::run<float>(int, const double *, const double *,
                                const double *, double *, double *, hipStream_t);
template int group_stages<float>(FcmGroup &, std::vector<char> *, hipStream_t);
template int set_fft_lds_attr<float>(const FftPlan &, const FftPlan &,
                                     const FftPlan &);
template int interp_blocks<float>(const FcmImpl &);
}  // namespace fs
