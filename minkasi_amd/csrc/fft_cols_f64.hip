// Column passes of the 2^11-point-row FFT engine in double (fft_cols.h).
#include "fft_cols.h"

namespace mkfft {
template void launch_cols_fwd<double>(int, int, const Seg*, int, int64_t, const void*, cx<double>*, const cx<double>*,
                                     const cx<double>*, const cx<double>*, int, hipStream_t);
template void launch_cols_inv<double>(int, int, const Seg*, int, int64_t, const cx<double>*, void*, const cx<double>*,
                                     const cx<double>*, const cx<double>*, hipStream_t);
}  // namespace mkfft
