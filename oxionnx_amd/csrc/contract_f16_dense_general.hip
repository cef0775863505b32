// MFMA contraction kernels, f16, dense operands, general epilogue.
#define OHIP_OP Op::F16
#define OHIP_OUT _Float16
#define OHIP_SUFFIX f16
#define OHIP_PART 4
#include "contract.inc"
