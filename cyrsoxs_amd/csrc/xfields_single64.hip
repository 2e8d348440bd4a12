// Fields + X FFT kernel (xfields.hpp), FP64, single mode.
#include "xfields.hpp"

namespace cyr {

template cyr_status launch_xfields<double, kXSingle>(PolxArgs<double>, const void *, int, int, bool, hipStream_t);

}  // namespace cyr
