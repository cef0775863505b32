// MFMA contraction kernels, f16, implicit im2col, pixels on Y (NHWC outputs).
#define OHIP_OP Op::F16
#define OHIP_OUT _Float16
#define OHIP_SUFFIX f16
#define OHIP_PART 3
#include "contract.inc"
