// Queue kernels of bf16 weights.
#include "gemm_queue.h"

template void launch_queue<false, MODE_BF>(const void*, const void*, const void*, float*, int, int, int, int, int,
                                       const Epilogue&, hipStream_t);
template void launch_queue<false, MODE_BF_GLU>(const void*, const void*, const void*, float*, int, int, int, int, int,
                                       const Epilogue&, hipStream_t);
template void launch_queue<false, MODE_BF_POST>(const void*, const void*, const void*, float*, int, int, int, int, int,
                                       const Epilogue&, hipStream_t);
template void launch_queue_rows<MODE_BF>(const void*, const void*, float*, int, int, int, int, int, const Epilogue&,
                                     hipStream_t);
template void launch_queue_rows<MODE_BF_GLU>(const void*, const void*, float*, int, int, int, int, int, const Epilogue&,
                                     hipStream_t);
template void launch_queue_rows<MODE_BF_POST>(const void*, const void*, float*, int, int, int, int, int, const Epilogue&,
                                     hipStream_t);
