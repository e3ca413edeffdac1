// tfgfa_fwd_f16.hip - the fp16 instances of the forward kernels (tfgfa_fwd.hip), a translation unit
// of their own.
#define TFGFA_FWD_F16_UNIT
#include "tfgfa_fwd.hip"
