// The convolution by stationary row with the whole weight in LDS (rows_hold.hip).
#pragma once
#include "conv_wave.h"

// Does its kernel take this call, which can go by rows, on a grid of ntiles tiles?
bool sph_rows_hold_ok(sph_dtype dt, const ConvArgs &a, int nwtot, int ntiles);
int sph_rows_hold_launch(sph_dtype dt, const ConvArgs &a, hipStream_t st);
