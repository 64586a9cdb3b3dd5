#include "chs_fft_impl.h"

namespace chs {

template void launch_fft_s<double>(cx<double>*, int, int, long, int, long, const Radices&, const cx<double>*, double, hipStream_t);
template void launch_fft_x<double>(bool, const double*, cx<double>*, double*, int, long, const Radices&, const cx<double>*,
                                  const cx<double>*, double, hipStream_t);
template void tune_transforms<double>(int, int, int, int, bool, cx<double>*, cx<double>*, const cx<double>*,
                                      const cx<double>*, const cx<double>*, const cx<double>*);

}  // namespace chs
