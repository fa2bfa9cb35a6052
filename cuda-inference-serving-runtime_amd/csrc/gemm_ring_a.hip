#include "gemm_ring.inc"

// tiles are named by rows * 1000 + columns
int cisr_ring_launch_a(const RingArgs& a, int tile, int mode, hipStream_t stream) {
    switch (tile) {
        case 288256: return ring_modes<9, 4, 2, 4, 2>(a, mode, stream);
        case 256256: return ring_modes<8, 4, 2, 4, 2>(a, mode, stream);
        case 224256: return ring_modes<7, 4, 2, 4, 2>(a, mode, stream);
    }
    return (int)hipErrorInvalidValue;
}
