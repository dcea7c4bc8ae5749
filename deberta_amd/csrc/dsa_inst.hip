// dsa_inst.hip — the attention kernels of one element type DSA_T and head dim
// DSA_D (macros of the build): see dsa_launch.h.
#include "dsa_launch.h"

namespace dsa {
namespace host {
template int fwd_mask<DSA_T, DSA_D>(const FwdParams&, int, hipStream_t);
template int launch_bwd<DSA_T, DSA_D>(const dsa_bwd_args*, const WsLayout&, int, hipStream_t);
}  // namespace host
}  // namespace dsa
