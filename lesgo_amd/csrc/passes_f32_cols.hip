// Column-pass launchers instantiated for float.
#include "passes_impl.hpp"

namespace lg {

template void launch_cols<float, -1>(KernelTimer&, ColArgs<float>&, int, int, int, int, hipStream_t,
                                   const PassChoice*);
template void launch_cols<float, +1>(KernelTimer&, ColArgs<float>&, int, int, int, int, hipStream_t,
                                   const PassChoice*);

}  // namespace lg
