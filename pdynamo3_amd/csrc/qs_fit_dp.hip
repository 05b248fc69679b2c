// Electron-fit integral kernels of the pair classes dp.
#define QS_FIT_KERNELS
#include "qs_fit_kernels.h"

namespace qs {

template void launch_fit<2, 1, 0>(const FitLaunch &, const PairItem *, int);
template void launch_fit<2, 1, 1>(const FitLaunch &, const PairItem *, int);
template void launch_fit<2, 1, 2>(const FitLaunch &, const PairItem *, int);

}  // namespace qs
