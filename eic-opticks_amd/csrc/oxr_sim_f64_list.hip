// oxr_sim_f64_list.hip -- simulate kernels with double-precision roots and list-node support
#include "oxr_sim.h"

namespace oxl {
template hipError_t launch_simulate_plain<true, true>(hipStream_t, const oxd::Params&, dim3, dim3, size_t, int, int);
template hipError_t launch_simulate_persist<true, true>(hipStream_t, const oxd::Params&, dim3, dim3, size_t, bool, int);
template const void* persist_kernel<true, true>(bool, int);
} // namespace oxl
