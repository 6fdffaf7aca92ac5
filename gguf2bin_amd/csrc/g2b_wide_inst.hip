// g2b_wide_inst.hip - one (KV format, head_dim) of k_wide's launchers.  The
// build compiles this file once per combination with -DG2B_FMT=<0|1>
// -DG2B_HD=<64|128|256>.
#include "g2b_wide.h"

#if !defined(G2B_FMT) || !defined(G2B_HD)
#error "g2b_wide_inst.hip needs -DG2B_FMT and -DG2B_HD"
#endif

namespace g2b {
template hipError_t launch_wide_hd<G2B_FMT, G2B_HD>(const DecodeParams &, int, hipStream_t);
template int wide_occupancy_hd<G2B_FMT, G2B_HD>(const ShapeDev &);
}  // namespace g2b
