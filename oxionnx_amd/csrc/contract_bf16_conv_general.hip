// MFMA contraction kernels, bf16, implicit im2col, pixels on X (NCHW outputs), general epilogue.
#define OHIP_OP Op::BF16
#define OHIP_OUT __bf16
#define OHIP_SUFFIX bf16
#define OHIP_PART 5
#include "contract.inc"
