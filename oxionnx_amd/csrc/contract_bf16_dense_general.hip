// MFMA contraction kernels, bf16, dense operands, general epilogue.
#define OHIP_OP Op::BF16
#define OHIP_OUT __bf16
#define OHIP_SUFFIX bf16
#define OHIP_PART 4
#include "contract.inc"
