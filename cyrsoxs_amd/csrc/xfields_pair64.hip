// Fields + X FFT kernel (xfields.hpp), FP64, pair mode.
#include "xfields.hpp"

namespace cyr {

template cyr_status launch_xfields<double, kXPair>(PolxArgs<double>, const void *, int, int, bool, hipStream_t);

}  // namespace cyr
