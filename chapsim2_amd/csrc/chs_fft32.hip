#include "chs_fft_impl.h"

namespace chs {

template void launch_fft_s<float>(cx<float>*, int, int, long, int, long, const Radices&, const cx<float>*, float, hipStream_t);
template void launch_fft_x<float>(bool, const float*, cx<float>*, float*, int, long, const Radices&, const cx<float>*,
                                  const cx<float>*, float, hipStream_t);

}  // namespace chs
