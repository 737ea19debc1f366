// Column-pass launchers instantiated for double.
#include "passes_impl.hpp"

namespace lg {

template void launch_cols<double, -1>(KernelTimer&, ColArgs<double>&, int, int, int, int, hipStream_t,
                                   const PassChoice*);
template void launch_cols<double, +1>(KernelTimer&, ColArgs<double>&, int, int, int, int, hipStream_t,
                                   const PassChoice*);

std::vector<std::pair<int, int>> pass_splits(int N) { return splits_for(N); }

}  // namespace lg
