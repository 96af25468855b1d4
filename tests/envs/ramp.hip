// Instantiates and registers the test-only envs of ramp.h in the test env library.
#include "mg/device/env_kernels.h"
#include "ramp.h"

MG_DEFINE_ENV(Ramp1)
MG_DEFINE_ENV(Ramp3)
MG_DEFINE_ENV(Ramp15)
MG_DEFINE_ENV(Ramp33)
MG_DEFINE_ENV(Ramp63)
