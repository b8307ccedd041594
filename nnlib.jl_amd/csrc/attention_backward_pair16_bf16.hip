// Instantiation of the 16-bit attention gradient in one kernel per (head, batch) pair: bf16.
#define BWD_T BF16
#define PAIR_ENTRY launch_bwd_pair16_bf16
#include "attention_backward_pair16.inc"
