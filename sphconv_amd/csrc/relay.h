// The grouped convolution with the weight held in the compute units' registers (relay.hip).
#pragma once
#include "conv_wave.h"

// Does the relay kernel take this call, on a grid of ntiles tiles?  (Rows and weight fit, and the grid is long enough.)
bool sph_relay_ok(sph_dtype dt, const ConvArgs &a, int nwtot, int ntiles);
int sph_relay_launch(sph_dtype dt, const ConvArgs &a, int nwtot, int ntiles, hipStream_t st);
