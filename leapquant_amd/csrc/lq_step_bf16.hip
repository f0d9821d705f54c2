// The kernels and launches of lq_step.hip for calls in which a gate parameter (A_log, dt_bias) is held in bf16.
#define LQ_GATE_BF16 1
#include "lq_step.hip"
