#include "gemm_ring.inc"

// tiles are named by rows * 1000 + columns
int cisr_ring_launch_d(const RingArgs& a, int tile, int mode, hipStream_t stream) {
    switch (tile) {
        case 160128: return ring_modes<5, 2, 2, 4, 3>(a, mode, stream);
        case 128128: return ring_modes<4, 2, 2, 4, 4>(a, mode, stream);
        case 96128: return ring_modes<3, 2, 2, 4, 4>(a, mode, stream);
        case 64128: return ring_modes<2, 2, 2, 4, 5>(a, mode, stream);
        case 128064: return ring_modes<2, 2, 4, 2, 3>(a, mode, stream);
        case 64064: return ring_modes<1, 2, 4, 2, 6>(a, mode, stream);
        case 64032: return ring_modes<1, 2, 4, 1, 10>(a, mode, stream);
    }
    return (int)hipErrorInvalidValue;
}
