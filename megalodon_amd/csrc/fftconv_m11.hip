// The convolution's transforms of 2048 complex points (rows of up to 4096 steps).
#define MEGA_FFTCONV_LOGM 11
#include "fftconv_rows.hpp"
