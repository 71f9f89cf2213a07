#include "tq_decode_kernel.h"

int tq_decode_launch_d64(int ipbk, int ipbv, dim3 grid, hipStream_t s, const TqDecodeArgs &a) {
    switch (ipbk) {
        case 4: return launch_decode<64, 4>(ipbv, grid, s, a);
        case 2: return launch_decode<64, 2>(ipbv, grid, s, a);
        case 1: return launch_decode<64, 1>(ipbv, grid, s, a);
        default: return TQ_ERR_BITS;
    }
}
