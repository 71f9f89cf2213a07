#include "tq_decode_kernel.h"

int tq_decode_launch_d128_narrow(int ipbk, int ipbv, dim3 grid, hipStream_t s, const TqDecodeArgs &a) {
    return ipbk == 8 ? launch_decode<128, 8>(ipbv, grid, s, a) : launch_decode<128, 4>(ipbv, grid, s, a);
}
