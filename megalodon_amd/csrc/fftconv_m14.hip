// The convolution's transforms of 16384 complex points (rows of up to 32768 steps).
#define MEGA_FFTCONV_LOGM 14
#include "fftconv_rows.hpp"
