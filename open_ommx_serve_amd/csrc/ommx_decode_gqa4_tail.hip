// The kernels of ommx_decode_gqa4.hip with the tail rows attended in the same launch (ommx_decode_tail.h).
#define OMMX_GQA4_LAUNCH launch_decode_gqa4_tail
#include "ommx_decode_gqa4.hip"
