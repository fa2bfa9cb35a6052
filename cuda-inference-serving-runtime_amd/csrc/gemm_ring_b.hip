#include "gemm_ring.inc"

// tiles are named by rows * 1000 + columns
int cisr_ring_launch_b(const RingArgs& a, int tile, int mode, hipStream_t stream) {
    switch (tile) {
        case 192256: return ring_modes<6, 4, 2, 4, 2>(a, mode, stream);
        case 160256: return ring_modes<5, 4, 2, 4, 3>(a, mode, stream);
        case 128256: return ring_modes<4, 4, 2, 4, 3>(a, mode, stream);
        case 96256: return ring_modes<3, 4, 2, 4, 3>(a, mode, stream);
    }
    return (int)hipErrorInvalidValue;
}
