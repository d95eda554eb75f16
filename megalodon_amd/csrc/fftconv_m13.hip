// The convolution's transforms of 8192 complex points (rows of up to 16384 steps).
#define MEGA_FFTCONV_LOGM 13
#include "fftconv_rows.hpp"
