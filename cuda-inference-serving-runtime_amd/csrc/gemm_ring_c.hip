#include "gemm_ring.inc"

// tiles are named by rows * 1000 + columns
int cisr_ring_launch_c(const RingArgs& a, int tile, int mode, hipStream_t stream) {
    switch (tile) {
        case 64256: return ring_modes<2, 4, 2, 4, 3>(a, mode, stream);
        case 256128: return ring_modes<8, 2, 2, 4, 3>(a, mode, stream);
        case 224128: return ring_modes<7, 2, 2, 4, 3>(a, mode, stream);
        case 192128: return ring_modes<6, 2, 2, 4, 3>(a, mode, stream);
    }
    return (int)hipErrorInvalidValue;
}
