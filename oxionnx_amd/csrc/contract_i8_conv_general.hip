// MFMA contraction kernels, i8, implicit im2col, pixels on X (NCHW outputs), general epilogue.
#define OHIP_OP Op::I8
#define OHIP_OUT void
#define OHIP_SUFFIX i8
#define OHIP_PART 5
#define OHIP_QUANT 1
#include "contract.inc"
