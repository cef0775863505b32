// MFMA contraction kernels, f32, implicit im2col, pixels on X (NCHW outputs), general epilogue.
#define OHIP_OP Op::F32
#define OHIP_OUT float
#define OHIP_SUFFIX f32
#define OHIP_PART 5
#include "contract.inc"
