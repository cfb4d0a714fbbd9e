// olx_mixprop1.hip -- the mixed-radix propagation passes with QM = 1 (mixprop.hpp).
#define OLX_MIXPROP_QM 1
#include "mixprop.hpp"
