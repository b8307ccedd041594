// Instantiation of the 16-bit attention gradient in one kernel per (head, batch) pair: f16.
#define BWD_T F16
#define PAIR_ENTRY launch_bwd_pair16_f16
#include "attention_backward_pair16.inc"
