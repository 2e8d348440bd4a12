// Fields + X FFT kernels in FP64 (xfields.hpp).
#include "xfields.hpp"

namespace cyr {

template cyr_status launch_ebasis_polx<double>(PolxArgs<double>, const void *, int, int, bool, hipStream_t);
template cyr_status launch_mbasis_xfields<double>(PolxArgs<double>, bool, const void *, int, int, bool, hipStream_t);

}  // namespace cyr
