// Fields + X FFT kernel (xfields.hpp), FP32, pair mode.
#include "xfields.hpp"

namespace cyr {

template cyr_status launch_xfields<float, kXPair>(PolxArgs<float>, const void *, int, int, bool, hipStream_t);

}  // namespace cyr
