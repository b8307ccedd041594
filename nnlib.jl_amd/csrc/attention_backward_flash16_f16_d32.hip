// Instantiation of the MFMA attention backward for f16, head dims up to 32.
#define BWD_T F16
#define BWD_D 32
#define BWD_ENTRY launch_bwd_flash16_f16_d32
#include "attention_backward_flash16.inc"
