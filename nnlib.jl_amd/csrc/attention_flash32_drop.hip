// Float32 forward kernels with fused dropout: attention_flash32.hip again, with the keep decisions (see there).
#define FLASH32_DROP 1
#include "attention_flash32.hip"
