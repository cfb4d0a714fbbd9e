// olx_mixprop2.hip -- the mixed-radix propagation passes with QM = 2 (mixprop.hpp).
#define OLX_MIXPROP_QM 2
#include "mixprop.hpp"
