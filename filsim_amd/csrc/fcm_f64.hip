// The mobility solve in FP64.
#include "fcm_run.hpp"

namespace fs {
template int FcmImpl::run<double>(int, const double *, const double *,
                                const double *, double *, double *, hipStream_t);
template int group_stages<double>(FcmGroup &, std::vector<char> *, hipStream_t);
template int set_fft_lds_attr<double>(const FftPlan &, const FftPlan &,
                                     const FftPlan &);
template int interp_blocks<double>(const FcmImpl &);
}  // namespace fs
