// fp16 instantiations of the 16-bit MFMA kernels (a translation unit of their own, compiled beside the bf16 ones).
#define LASP_MFMA_F16
#include "lasp_mfma.hip"
