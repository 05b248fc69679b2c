// Electron-fit integral kernels of the pair classes dd with s and p fit shells.
#define QS_FIT_KERNELS
#include "qs_fit_kernels.h"

namespace qs {

template void launch_fit<2, 2, 0>(const FitLaunch &, const PairItem *, int);
template void launch_fit<2, 2, 1>(const FitLaunch &, const PairItem *, int);

}  // namespace qs
