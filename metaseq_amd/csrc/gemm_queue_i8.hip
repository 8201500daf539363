// Queue kernels of int8 weights.
#include "gemm_queue.h"

template void launch_queue<true, MODE_PLAIN>(const void*, const void*, const void*, float*, int, int, int, int, int,
                                       const Epilogue&, hipStream_t);
template void launch_queue<true, MODE_QKV>(const void*, const void*, const void*, float*, int, int, int, int, int,
                                       const Epilogue&, hipStream_t);
