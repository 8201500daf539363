// Queue kernels of fp16 weights.
#include "gemm_queue.h"

template void launch_queue<false, MODE_PLAIN>(const void*, const void*, const void*, float*, int, int, int, int, int,
                                       const Epilogue&, hipStream_t);
template void launch_queue<false, MODE_QKV>(const void*, const void*, const void*, float*, int, int, int, int, int,
                                       const Epilogue&, hipStream_t);
template void launch_queue_rows<MODE_PLAIN>(const void*, const void*, float*, int, int, int, int, int, const Epilogue&,
                                     hipStream_t);
template void launch_queue_rows<MODE_QKV>(const void*, const void*, float*, int, int, int, int, int, const Epilogue&,
                                     hipStream_t);
