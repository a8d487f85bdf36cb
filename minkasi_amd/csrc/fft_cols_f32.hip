// Column passes of the 2^11-point-row FFT engine in float (fft_cols.h).
#include "fft_cols.h"

namespace mkfft {
template void launch_cols_fwd<float>(int, int, const Seg*, int, int64_t, const void*, cx<float>*, const cx<float>*,
                                     const cx<float>*, const cx<float>*, int, hipStream_t);
template void launch_cols_inv<float>(int, int, const Seg*, int, int64_t, const cx<float>*, void*, const cx<float>*,
                                     const cx<float>*, const cx<float>*, hipStream_t);
}  // namespace mkfft
