#include "tq_decode_kernel.h"

int tq_decode_launch_d128_wide(int ipbk, int ipbv, dim3 grid, hipStream_t s, const TqDecodeArgs &a) {
    return ipbk == 2 ? launch_decode<128, 2>(ipbv, grid, s, a) : launch_decode<128, 1>(ipbv, grid, s, a);
}
