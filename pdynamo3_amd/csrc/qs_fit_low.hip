// Electron-fit integral kernels of the pair classes ss, ps, pp and ds.
#define QS_FIT_KERNELS
#include "qs_fit_kernels.h"

namespace qs {

template void launch_fit<0, 0, 0>(const FitLaunch &, const PairItem *, int);
template void launch_fit<0, 0, 1>(const FitLaunch &, const PairItem *, int);
template void launch_fit<0, 0, 2>(const FitLaunch &, const PairItem *, int);
template void launch_fit<1, 0, 0>(const FitLaunch &, const PairItem *, int);
template void launch_fit<1, 0, 1>(const FitLaunch &, const PairItem *, int);
template void launch_fit<1, 0, 2>(const FitLaunch &, const PairItem *, int);
template void launch_fit<1, 1, 0>(const FitLaunch &, const PairItem *, int);
template void launch_fit<1, 1, 1>(const FitLaunch &, const PairItem *, int);
template void launch_fit<1, 1, 2>(const FitLaunch &, const PairItem *, int);
template void launch_fit<2, 0, 0>(const FitLaunch &, const PairItem *, int);
template void launch_fit<2, 0, 1>(const FitLaunch &, const PairItem *, int);
template void launch_fit<2, 0, 2>(const FitLaunch &, const PairItem *, int);

}  // namespace qs
