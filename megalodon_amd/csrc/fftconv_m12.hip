// The convolution's transforms of 4096 complex points (rows of up to 8192 steps).
#define MEGA_FFTCONV_LOGM 12
#include "fftconv_rows.hpp"
