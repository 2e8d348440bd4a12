// Fields + X FFT kernels in FP32 (xfields.hpp).
#include "xfields.hpp"

namespace cyr {

template cyr_status launch_ebasis_polx<float>(PolxArgs<float>, const void *, int, int, bool, hipStream_t);
template cyr_status launch_mbasis_xfields<float>(PolxArgs<float>, bool, const void *, int, int, bool, hipStream_t);

}  // namespace cyr
