// MFMA contraction kernels, f16, implicit im2col, pixels on X (NCHW outputs), general epilogue.
#define OHIP_OP Op::F16
#define OHIP_OUT _Float16
#define OHIP_SUFFIX f16
#define OHIP_PART 5
#include "contract.inc"
