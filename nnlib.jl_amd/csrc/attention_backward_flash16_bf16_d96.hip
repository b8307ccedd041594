// Instantiation of the MFMA attention backward for bf16, head dims up to 96.
#define BWD_T BF16
#define BWD_D 96
#define BWD_ENTRY launch_bwd_flash16_bf16_d96
#include "attention_backward_flash16.inc"
