// Split type-1 path, FP64: the term kernel.
#include "sg4_split.h"

namespace sg4 {

__global__ __launch_bounds__(NT) void k_hpsi_t1s_f64(KArgs a, KMats<double> km) { split_items<double, false>(a, km); }
__global__ __launch_bounds__(NT) void k_hpsi_t1s_out_f64(KArgs a, KMats<double> km) { split_items<double, true>(a, km); }

}  // namespace sg4
