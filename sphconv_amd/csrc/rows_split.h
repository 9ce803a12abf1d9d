// The convolution by stationary row with a row's offsets shared by the waves of a workgroup (rows_split.hip).
#pragma once
#include "conv_wave.h"

// Does one of its kernels take this call, which can go by rows, on a grid of ntiles tiles?
bool sph_rows_split_ok(sph_dtype dt, const ConvArgs &a, int nwtot, int ntiles);
int sph_rows_split_launch(sph_dtype dt, const ConvArgs &a, int nwtot, int ntiles, hipStream_t st);
