// The direct anisotropic embedding kernel behind a condition on the device: nothing is written where *taken is not 0 (another kernel
// of the same call has done the work).  taken = NULL: unconditional.
#pragma once
#include <stdint.h>

int proteus_we_aniso_direct(const float* coordsA, const float* coordsB, int coords_layout,
                            const float* cb_magnitudes, const float* wavenumbers, const uint8_t* mask,
                            float* out, float* d_cb, float* d_k, int Z, int N, int K, int tuning, const int* taken, void* stream);
