// MFMA contraction kernels, f32, dense operands, general epilogue.
#define OHIP_OP Op::F32
#define OHIP_OUT float
#define OHIP_SUFFIX f32
#define OHIP_PART 4
#include "contract.inc"
