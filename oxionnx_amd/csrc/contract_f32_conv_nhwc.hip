// MFMA contraction kernels, f32, implicit im2col, pixels on Y (NHWC outputs).
#define OHIP_OP Op::F32
#define OHIP_OUT float
#define OHIP_SUFFIX f32
#define OHIP_PART 3
#include "contract.inc"
